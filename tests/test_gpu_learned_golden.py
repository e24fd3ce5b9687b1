"""The network's losses and gradients, bit for bit as recorded.

tests/golden/mpnn_gradients.npz (tests/golden/make_mpnn_golden.py) holds what
one batch gives.  A gradient whose exact value is zero (the decoder's bias:
the output is made mean-free) is the rounding of its sum alone, and Adam's
first step, lr sign(g), makes whole steps of it, so a sum in another order
would train another network from the same data.
"""
import importlib.util
import os

import numpy as np
import pytest

from conftest import golden

pytest.importorskip("flowsolversourcecode_amd")
pytestmark = pytest.mark.gpu

_spec = importlib.util.spec_from_file_location(
    "make_mpnn_golden", os.path.join(os.path.dirname(__file__), "golden", "make_mpnn_golden.py"))
mg = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(mg)


@pytest.mark.parametrize("name", list(mg.CASES))
def test_gradient_is_the_recorded_one(name):
    g = golden("mpnn_gradients.npz")
    loss, grad = mg.run(name)
    want = g[name + "_grad"]
    assert np.array_equal(grad, want), np.flatnonzero(grad != want)[:8]
    assert loss == g[name + "_loss"]
