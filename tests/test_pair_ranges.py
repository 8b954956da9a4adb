"""The pair passes' loops at totals up to 2^32 - 1 candidates, by host arithmetic
alone (tests/cpp/pair_ranges_check.hip): with 32-bit candidate indices the step
past the last candidate wrapped for totals above 2^32 - 2^22 and the loop never
ended."""
import os
import subprocess

from voxelizer_amd import build as B

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_block_of_candidates_is_taken_once(tmp_path):
    exe = str(tmp_path / "pair_ranges_check")
    subprocess.run([B.hipcc(), "-O1", "-std=c++17", "-x", "hip", "--offload-host-only",
                    f"--offload-arch={B.ARCH}", "-I", B.CSRC, "-o", exe,
                    os.path.join(HERE, "cpp", "pair_ranges_check.hip")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
