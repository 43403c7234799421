import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on the GPU box)")


def pytest_collection_modifyitems(config, items):
    import torch

    if torch.cuda.is_available():
        return
    skip = pytest.mark.skip(reason="no GPU in this container")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)


@pytest.fixture(scope="session")
def dev():
    import torch

    return torch.device("cuda", 0)


@pytest.fixture(params=[-1, 0, 1], ids=["chosen-build", "three-per-cu", "two-per-cu"])
def fp8_build(request):
    """Every test that asks for it runs with the GEMM's kernel chosen by size (for small launches the one that splits K)
    and with each build of the fp8 main loop, which serve the large launches."""
    from nunchaku_rocm_amd.ops import gemm as G

    G.set_fp8_loop_variant(request.param)
    yield request.param
    G.set_fp8_loop_variant(-1)
