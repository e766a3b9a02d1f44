import gc
import os
import sys

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)
HERE = os.path.dirname(os.path.abspath(__file__))
if HERE not in sys.path:
    sys.path.insert(0, HERE)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a ROCm GPU (MI355X) and the built HIP library")


def pytest_collection_modifyitems(config, items):
    if torch.cuda.is_available():
        return
    skip = pytest.mark.skip(reason="no ROCm GPU visible")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)


@pytest.fixture(autouse=True)
def _seed():
    torch.manual_seed(0)


@pytest.fixture(autouse=True, scope="module")
def _no_garbage_between_modules():
    """A module's cyclic garbage (engines that hold HIP graphs) goes before the next module's tests, which
    capture graphs of their own: destroying a graph inside a capture ends the process."""
    yield
    gc.collect()


def pytest_terminal_summary(terminalreporter):
    from helpers import RECORDS

    if RECORDS:
        terminalreporter.section("parity figures")
        for line in RECORDS:
            terminalreporter.write_line(line)
