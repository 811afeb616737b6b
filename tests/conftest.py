import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP step library)")


def gpu_available():
    try:
        import torch  # noqa: F401  (device discovery only)
        return torch.cuda.is_available()
    except Exception:
        return False


@pytest.fixture(scope="session")
def ref_available():
    from oracle import ref
    if not ref.available():
        pytest.skip("reference harness not built (make -C oracle)")
    return True


@pytest.hookimpl(wrapper=True)
def pytest_runtest_call(item):
    """A test that compares with the reference harness says so, and is skipped, where the harness cannot be built."""
    from oracle import ref
    try:
        return (yield)
    except ref.HarnessMissing as e:
        pytest.skip(str(e))
