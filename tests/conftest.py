import gc
import importlib
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP kernels through the C ABI)")


def pytest_runtest_setup(item):
    # objects that earlier tests left in reference cycles give their device memory back here, not in
    # the middle of a test's graph capture (a free while a stream is captured invalidates the capture)
    if item.get_closest_marker("gpu"):
        gc.collect()


@pytest.fixture(scope="session")
def vsc():
    """The product package (directory name contains hyphens)."""
    return importlib.import_module("video-stream-consistency_amd")


@pytest.fixture(scope="session")
def orc():
    """The CPU oracle (test infrastructure)."""
    from oracle import oracle
    oracle.lib()
    return oracle


@pytest.fixture(scope="session")
def cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


@pytest.fixture
def rng():
    return np.random.default_rng(1234)
