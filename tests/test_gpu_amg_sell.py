"""One multigrid cycle in numpy (test_gpu_amg_dense.py, and its tolerances)
against the device with every large level in sliced ELL: columns as 16-bit
offsets on a mesh numbered row by row, as 32-bit columns on the same mesh
numbered at random, whose second level has neighbours more than 32767 rows
apart.
"""
import numpy as np
import pytest

from test_gpu_amg_dense import full_cycle, run

pytest.importorskip("flowsolversourcecode_amd")
pytestmark = pytest.mark.gpu


def grid(nx, ny, shuffled):
    n = nx * ny
    rng = np.random.default_rng(3)
    name = rng.permutation(n) if shuffled else np.arange(n)
    c = np.arange(n)
    i, j = c % nx, c // nx
    nbr = np.zeros((4, n), np.int32)
    anb = np.zeros((4, n))
    wx, wy = -rng.uniform(0.5, 1.5, n), -rng.uniform(0.5, 1.5, n)  # of the faces towards +x and +y
    faces = [(i > 0, c - 1, wx[c - 1]), (i < nx - 1, (c + 1) % n, wx), (j > 0, c - nx, wy[c - nx]),
             (j < ny - 1, (c + nx) % n, wy)]
    for s, (ok, k, a) in enumerate(faces):
        nbr[s, name] = np.where(ok, name[k] + 1, 0)
        anb[s, name] = np.where(ok, a, 0.0)
    ac = 0.05 - anb.sum(0)
    return nbr, np.full(n, 4, np.int32), ac, anb, rng.standard_normal(n)


@pytest.mark.parametrize("shape,shuffled", [((41, 37), False), ((500, 400), False), ((700, 500), True)], ids=str)
@pytest.mark.parametrize("fp32", [0, 1])
def test_one_cycle_is_numpys(shape, shuffled, fp32):
    system = grid(*shape, shuffled)
    opts = {"mg_sell_rows": 1, "mg_tail_cells": 100, "mg_fp32": fp32}
    dphi, levels = run(system, opts)
    A = levels[1].A.tocoo()
    assert (np.abs(A.row - A.col).max() > 32767) == shuffled
    ts = next(l for l in range(1, len(levels)) if levels[l].n <= 100)
    want = full_cycle(levels, ts, system[4], opts, -16)
    np.testing.assert_allclose(dphi, want, rtol=0, atol=(1e-4 if fp32 else 1e-11) * np.abs(want).max())
