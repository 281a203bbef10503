import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on the GPU box)")


@pytest.fixture(params=[-1, 0], ids=["chosen", "256x256"])
def kernel(request):
    """The tiled GEMM kernel that a problem goes to by itself (at most tests' sizes one of the smaller tiles), and the 256 x 256 one."""
    import catccos_amd as cc
    cc.set_option("gemm_kernel", request.param)
    yield request.param
    cc.set_option("gemm_kernel", -1)


def _has_gpu():
    try:
        import torch
        return torch.cuda.is_available()
    except Exception:
        return False


def pytest_collection_modifyitems(config, items):
    if _has_gpu():
        return
    skip = pytest.mark.skip(reason="no GPU visible")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)
