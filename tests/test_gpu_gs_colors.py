"""Multicolour Gauss-Seidel against the same sweeps in numpy, bit for bit:
systems swept in cell order and systems copied into colour order (three colours
and more, 800000 slots and more), just below and above that line.

The colours are first fit in cell order; a cell's terms are subtracted from its
right-hand side in slot order.  One iteration sweeps the colours up and down.
"""
import numpy as np
import pytest

from test_gpu_ilu_order import graph

fs = pytest.importorskip("flowsolversourcecode_amd")
pytestmark = pytest.mark.gpu


def colors(nbr):
    w, n = nbr.shape
    color = [-1] * n
    rows = (nbr.T - 1).tolist()
    for i in range(n):
        used = {color[k] for k in rows[i] if k >= 0}
        c = 0
        while c in used:
            c += 1
        color[i] = c
    return np.array(color)


def sweep(nbr, ac, anb, bc, x, cells):
    s = bc[cells].copy()
    for j in range(len(nbr)):
        k = nbr[j, cells] - 1
        s -= np.where(k >= 0, anb[j, cells] * x[np.maximum(k, 0)], 0.0)
    x[cells] = s / ac[cells]


@pytest.mark.parametrize("n,edges,w", [(900, 1500, 4), (199999, 330000, 4), (200000, 330000, 4), (160001, 360000, 5),
                                       (90001, 340000, 9)])
def test_sweeps_are_numpys(n, edges, w):
    nbr, nnbr, ac, anb, bc = graph(n, edges, w, 9)
    color = colors(nbr)
    nc = color.max() + 1
    assert nc >= 3
    m = fs.Mesh(nbr, nnbr)
    rc, f, dphi, res4, st = m.solve_equation("velx", np.zeros(n), 1e-30, 2, "sor", 0, ac, anb, bc)
    x = np.zeros(n)
    lists = [np.nonzero(color == c)[0] for c in range(nc)]
    for _ in range(2):
        for c in list(range(nc)) + list(range(nc - 2, -1, -1)):
            sweep(nbr, ac, anb, bc, x, lists[c])
    assert np.array_equal(dphi, x), np.abs(dphi - x).max()
