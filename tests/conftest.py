import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

REFOUT_DIR = os.path.join(ROOT, "tests", "golden")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP kernels)")


def pytest_collection_modifyitems(config, items):
    # Announce each GPU test before it runs so a failing box names the case.
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(pytest.mark.timeout(300))


@pytest.fixture(scope="session")
def gpu():
    import torch

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    torch.cuda.set_device(0)
    return 0


@pytest.fixture(scope="module", autouse=True)
def _oracle_blas_threads(request):
    """The oracle's golden-run chains are unconverged plain recurrences, whose last
    printed digit depends on how the BLAS splits a dot product over threads: one
    thread gives the same digits whatever the number of CPUs."""
    if request.module.__name__ != "test_refout_oracle":
        yield
        return
    import numpy  # noqa: F401  (the BLAS to limit)
    import scipy.linalg  # noqa: F401
    from threadpoolctl import threadpool_limits

    with threadpool_limits(1, user_api="blas"):
        yield
