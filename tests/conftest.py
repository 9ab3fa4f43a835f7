import os
import sys

import pytest


ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "accelerated-model-architectures_amd")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


def pytest_collection_modifyitems(config, items):
    import torch

    if torch.cuda.is_available():
        return
    skip = pytest.mark.skip(reason="no GPU visible")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)


@pytest.fixture(params=["chosen", "256 x 256"])
def either_tile(request, monkeypatch):
    """the grouped GEMMs by the dispatch rule, and by the 256 x 256 kernels whatever the rule says"""
    from xma.rocm import ops

    if request.param == "256 x 256":
        monkeypatch.setattr(ops, "FEW_ROWS_MAX", 0)
