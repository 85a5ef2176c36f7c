"""pytest configuration: import paths and the `gpu` marker."""

import gc
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
for p in (ROOT, ROOT / "rldx-1_amd"):
    if str(p) not in sys.path:
        sys.path.insert(0, str(p))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a ROCm GPU (MI355X / gfx950)")


@pytest.fixture(autouse=True)
def collect_before_gpu_tests(request):
    """Graphs of earlier tests that sit in reference cycles are freed here, not by
    a collection inside a test's own stream capture (where freeing one aborts)."""
    if request.node.get_closest_marker("gpu"):
        gc.collect()


@pytest.fixture(scope="session")
def dev():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU visible")
    return torch.device("cuda:0")
