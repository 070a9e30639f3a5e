import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "stickbreaking-attention_amd")):
    if p not in sys.path:
        sys.path.insert(0, p)


@pytest.fixture(params=["by size", "general"])
def kernels(request, monkeypatch):
    """By itself a call takes kernels by its size; problems as small as most tests' never reach the general forward and the two
    passes of the backward, which are asked for here."""
    from stickbreaking_attention import _native, _ops
    lib = _native.load()
    if request.param == "general":
        monkeypatch.setattr(_ops, "FORWARD_FLAGS", _native.FLAG_GENERAL_FORWARD)
        lib.sba_set_backward_form(1)
    yield request.param
    lib.sba_set_backward_form(0)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on the GPU box)")
