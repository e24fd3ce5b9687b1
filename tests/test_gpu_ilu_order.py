"""The ILU iteration and PBCG's D-ILU on graphs that reach every form of the
level schedule, against the oracle.

The schedule runs consecutive narrow levels (up to 2048 cells) in one
workgroup and a wider level as a launch of its own, with kernels for up to 4,
6 and 8 terms a cell and level launches for more.  Random graphs set the
widths and term counts a mesh would not: a chain (every level one cell), few
edges (the first levels thousands of cells wide, narrow ones after them), and
rows of up to 12 neighbours.  ILU iterates are the reference's bit for bit, so
the comparison is exact; PBCG's dots are summed in another order, so its
history agrees to 1e-10 over 5 iterations as in test_gpu_solve.py.
"""
import numpy as np
import pytest

import pyoracle as po

fs = pytest.importorskip("flowsolversourcecode_amd")
pytestmark = pytest.mark.gpu


def graph(n, edges, w, seed, chain=False):
    """n cells, about `edges` random couplings with at most w slots a row."""
    rng = np.random.default_rng(seed)
    pairs = rng.integers(0, n, (edges, 2))
    if chain:
        pairs = np.concatenate([np.stack([np.arange(n - 1), np.arange(1, n)], 1), pairs])
    pairs.sort(axis=1)
    keep = dict.fromkeys((int(a), int(b)) for a, b in pairs if a != b)
    rows = [[] for _ in range(n)]
    for a, b in keep:
        if len(rows[a]) < w and len(rows[b]) < w:
            rows[a].append(b)
            rows[b].append(a)
    nbr = np.zeros((w, n), np.int32)
    nnbr = np.zeros(n, np.int32)
    anb = np.zeros((w, n))
    for i, r in enumerate(rows):
        nnbr[i] = len(r)
        for s, k in enumerate(r):
            nbr[s, i] = k + 1
            anb[s, i] = -rng.uniform(0.2, 1.0)
    ac = 0.3 - anb.sum(0)
    return nbr, nnbr, ac, anb, rng.standard_normal(n)


GRAPHS = {
    "chain": (300, 0, 4, True),
    "one cell": (1, 0, 4, False),
    "narrow, 4 terms": (900, 1500, 4, True),
    "narrow, 6 terms": (3000, 7000, 6, True),
    "a level of 1024 and more": (5000, 6000, 4, False),
    "wide, then narrow": (30000, 36000, 5, False),
    "8 terms": (4000, 12000, 8, False),
    "more terms than the runs take": (6000, 30000, 12, False),
}


@pytest.mark.parametrize("name", GRAPHS)
def test_ilu_iterates_are_the_oracles(name):
    n, edges, w, chain = GRAPHS[name]
    nbr, nnbr, ac, anb, bc = graph(n, edges, w, 5, chain)
    m = fs.Mesh(nbr, nnbr)
    fit = np.linspace(-1.0, 1.0, n)
    for k in (1, 4):
        rc, f, dphi, res4, st = m.solve_equation("velx", fit, 0.0, k, "ilu", 0, ac, anb, bc)
        fo, do, _, _ = po.solve_equation(nbr, nnbr, ac, anb, bc, fit, 0.0, k, po.ILU, nf=1)
        assert np.array_equal(dphi, do) and np.array_equal(f, fo), np.abs(dphi - do).max()


@pytest.mark.parametrize("name", GRAPHS)
def test_pbcg_takes_the_same_diagonal(name):
    n, edges, w, chain = GRAPHS[name]
    nbr, nnbr, ac, anb, bc = graph(n, edges, w, 6, chain)
    m = fs.Mesh(nbr, nnbr)
    rc, f, dphi, res4, st = m.solve_equation("pressc", np.zeros(n), 1e-30, 5, "pbcg", 0, ac, anb, bc)
    fo, do, _, _ = po.solve_equation(nbr, nnbr, ac, anb, bc, np.zeros(n), 1e-30, 5, po.PBCG)
    np.testing.assert_allclose(dphi, do, rtol=0, atol=1e-10 * np.abs(do).max())
