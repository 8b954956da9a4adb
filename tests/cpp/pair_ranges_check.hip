// Host check of how the pair passes divide their candidates (vox_kernels.h), up
// to the largest total their 32-bit offsets hold: every block of 256 is taken
// exactly once and every loop ends.  Nothing runs on a device.
#include "vox_kernels.h"

#include <algorithm>
#include <cstdio>
#include <vector>

static int failures = 0;
static void expect(bool ok, const char *what, unsigned long long at) {
    if (ok) return;
    std::printf("FAIL %s (%llu)\n", what, at);
    failures++;
}

int main() {
    const uint32_t kMax = UINT32_MAX, kStep = 16384u * 256u;  // candidates a step of the largest grid
    const uint32_t totals[] = {0u,           1u,          255u,        256u,         257u,
                               kStep,        kStep + 1u,  4293918720u, kMax - kStep, kMax - kStep + 1u,
                               kMax - 256u,  kMax - 255u, kMax - 254u, kMax - 1u,    kMax};
    for (uint32_t total : totals) {
        const uint64_t want = ((uint64_t)total + 255u) / 256u;
        expect(vk::block_starts_size(total) == (size_t)want + 1u, "block_starts_size", total);
        expect(vk::graph_capacity(total) >= total, "graph_capacity", total);
        // The workgroups of a pass.
        const uint32_t blocks = (uint32_t)std::min<uint64_t>(std::max<uint64_t>(want, 1u), 16384u);
        std::vector<uint8_t> taken(want, 0);
        uint64_t steps = 0;
        for (uint32_t b = 0; b < blocks && steps <= want; b++)
            for (vk::CandRange r(b, blocks, total); r.more() && steps <= want; r.next(), steps++)
                taken[r.k]++;
        expect(steps == want, "steps of a pass", total);
        expect(std::count(taken.begin(), taken.end(), 1) == (long)want, "blocks taken once", total);
        // The block starts of three triangles that share the candidates.
        for (uint64_t cut : {(uint64_t)0, (uint64_t)total / 3u, (uint64_t)total / 256u * 256u}) {
            const uint32_t off[] = {0u, (uint32_t)cut, (uint32_t)cut, total};
            std::fill(taken.begin(), taken.end(), 0);
            for (int t = 0; t < 3; t++)
                for (uint32_t k = vk::cand_blocks(off[t]); k < vk::cand_blocks(off[t + 1]); k++) {
                    taken[k]++;
                    expect(off[t] <= k * 256ull && k * 256ull < off[t + 1], "block start", k);
                }
            expect(std::count(taken.begin(), taken.end(), 1) == (long)want, "starts set once", total);
        }
    }
    if (!failures) std::printf("ok\n");
    return failures != 0;
}
