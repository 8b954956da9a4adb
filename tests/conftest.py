import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device) and the built library")
    config.addinivalue_line("markers", "slow: large CPU work")


@pytest.fixture(scope="session")
def oracle():
    from oracle import oracle_py as O
    O.build()
    return O


@pytest.fixture(scope="session")
def gpu_ctx():
    """A library context on device 0.  No skip: on the GPU box a missing
    library or device is a failure."""
    import voxelizer_amd as va
    ctx = va.Context(0)
    yield ctx
    ctx.close()


@pytest.fixture(autouse=True)
def brick_shape_by_grid(request):
    """A test that sets a brick shape on the shared context leaves the grid's
    own choice to the tests after it, which run what users get."""
    ctx = request.getfixturevalue("gpu_ctx") if "gpu_ctx" in request.fixturenames else None
    yield
    if ctx is not None:
        for fcc in (False, True):
            ctx.set_brick_dims((0, 0, 0), fcc)
