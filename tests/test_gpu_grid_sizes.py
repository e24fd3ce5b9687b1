"""Reductions over grids of every form: padded to a multiple of eight
workgroups (64 workgroups and more), one row per thread, and rows strided by
the grid (above 8388608 rows).

A chain of cells with two slots a row, whose sums numpy forms.  A sum of n
non-negative terms in any order errs by at most n 2^-53 of itself.
"""
import numpy as np
import pytest

fs = pytest.importorskip("flowsolversourcecode_amd")
pytestmark = pytest.mark.gpu


def chain(n):
    i = np.arange(n, dtype=np.int32)
    nbr = np.stack([i, np.where(i + 1 < n, i + 2, 0)]).astype(np.int32)  # cell i-1, cell i+1 (1-based, 0 none)
    anb = np.where(nbr > 0, -1.0, 0.0)
    return nbr, np.full(n, 2, np.int32), np.full(n, 2.5), anb


def residual(ac, anb, bc, x):
    r = bc - ac * x
    r[1:] -= anb[0, 1:] * x[:-1]
    r[:-1] -= anb[1, :-1] * x[1:]
    return r


@pytest.mark.parametrize("n", [1, 256, 63 * 256, 64 * 256 + 1, 71 * 256 + 3, 8192 * 256 + 5, 32768 * 256 + 300])
@pytest.mark.parametrize("solver", ["sor", "bicgs", "cg"])
def test_sums_over_all_rows(n, solver):
    nbr, nnbr, ac, anb = chain(n)
    bc = np.random.default_rng(n).standard_normal(n)
    m = fs.Mesh(nbr, nnbr)
    rc, f, dphi, res4, st = m.solve_equation("velx", np.ones(n), 1e-30, 3, solver, 0, ac, anb, bc)
    first = np.abs(bc).sum()
    eps = max(n, 16) * 2.0**-53
    np.testing.assert_allclose(st["initial_l1"], first, rtol=eps)
    np.testing.assert_allclose(res4[0], first, rtol=eps)
    assert res4[1] == np.abs(bc).max()
    np.testing.assert_allclose(res4[2], np.sqrt((bc * bc).sum() / n), rtol=eps)
    # the Krylov residuals are updated, not formed from the iterate: they part
    # from it by the round-off of three iterations
    np.testing.assert_allclose(st["final_l1"], np.abs(residual(ac, anb, bc, dphi)).sum(), rtol=eps, atol=1e-13 * first)
