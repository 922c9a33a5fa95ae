import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run on the GPU box only)")


@pytest.fixture(scope="session")
def oracle():
    from oracle import oracle as orc
    return orc


@pytest.fixture(params=["as chosen", "without sliced kernels"])
def sliced(request, monkeypatch):
    """Once as the library chooses and once with the kernels it has for more tiles, which the same sizes went to before there were others for few."""
    if request.param != "as chosen":
        monkeypatch.setenv("NZHIP_GEMM_SLICES", "0")
        monkeypatch.setenv("NZHIP_CONV_SLICES", "0")


@pytest.fixture(params=["as chosen", "without sliced kernels", "without copies"])
def conv_ways(request, monkeypatch):
    """The same, and once with the window, gather and column kernels."""
    if request.param == "without sliced kernels":
        monkeypatch.setenv("NZHIP_GEMM_SLICES", "0")
        monkeypatch.setenv("NZHIP_CONV_SLICES", "0")
    elif request.param == "without copies":
        monkeypatch.setenv("NZHIP_CONV_CL", "0")
