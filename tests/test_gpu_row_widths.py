"""Rows of every width through the kernels that take a row's slots in batches
of 4, 6 or 8.

Empty slots add nothing and a row's terms are taken in slot order, so a
system whose table is padded with empty slots is the same system, and its
solves are the same bit for bit.  The multigrid's finest level spreads rows
above 8 slots over several lanes, which sums in another order: there the
widths end at 8.
"""
import numpy as np
import pytest

from test_gpu_ilu_order import graph

fs = pytest.importorskip("flowsolversourcecode_amd")
pytestmark = pytest.mark.gpu

N, W = 3001, 3


def padded(a, w):
    return np.concatenate([a, np.zeros((w - len(a),) + a.shape[1:], a.dtype)])


@pytest.mark.parametrize("solver,lmg,widths", [("sor", 0, (4, 5, 6, 7, 8, 9, 13)), ("pbcg", 0, (4, 5, 6, 7, 8, 9, 13)),
                                               ("cg", 2, (4, 5, 6, 7, 8)), ("bicgs", 2, (4, 5, 6, 7, 8))])
def test_empty_slots_change_nothing(solver, lmg, widths):
    nbr, nnbr, ac, anb, bc = graph(N, 5000, W, 8, chain=True)
    ref = None
    for w in (W,) + widths:
        m = fs.Mesh(padded(nbr, w), np.full(N, w, np.int32))
        rc, f, dphi, res4, st = m.solve_equation("pressc", np.zeros(N), 1e-30, 4, solver, lmg, ac, padded(anb, w), bc)
        r = bc - ac * dphi
        for s in range(W):
            k = nbr[s]
            r -= np.where(k > 0, anb[s] * dphi[np.maximum(k, 1) - 1], 0.0)
        # the Krylov solvers update their residual: it parts from the iterate's
        # by the round-off of four iterations
        np.testing.assert_allclose(st["final_l1"], np.abs(r).sum(), rtol=1e-12, atol=1e-12 * np.abs(bc).sum())
        if ref is None:
            ref = dphi
        assert np.array_equal(dphi, ref), (w, np.abs(dphi - ref).max())
