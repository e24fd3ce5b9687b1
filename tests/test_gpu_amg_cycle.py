"""Device AMG cycle variants against what the mathematics fixes.

The V-cycle's form (damped Jacobi or multicolour Gauss-Seidel smoothing,
fused restriction/prolongation kernels, the dense map of the small levels, the FP64
direct solve of the coarsest level, over-correction) changes the iterates but
not the solution: every variant must drive the true L1 residual of the system
below 1e-8 of its initial value, and on a non-singular system reach the sparse
direct solution to 1e-6 of its largest entry.  Systems of 15k cells give a
hierarchy with grid-wide levels above the tail threshold and tail levels
below it; mg_sell_rows = 1 puts every grid-wide coarse level in sliced ELL.
"""
import numpy as np
import pytest
import scipy.sparse.linalg as spl

import systems

fs = pytest.importorskip("flowsolversourcecode_amd")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def neumann():
    nbr, nnbr, ac, anb, bc = systems.pressure_like(32, 24, 20, 11, shift=0.0)
    return nbr, nnbr, ac, anb, bc, systems.sparse(nbr, nnbr, ac, anb)


@pytest.fixture(scope="module")
def shifted():
    nbr, nnbr, ac, anb, bc = systems.pressure_like(32, 24, 20, 12, shift=0.05)
    A = systems.sparse(nbr, nnbr, ac, anb)
    return nbr, nnbr, ac, anb, bc, A, spl.spsolve(A.tocsc(), bc)


VARIANTS = [
    {},
    {"mg_fp32": 1},
    {"mg_alpha": 1.0},
    {"mg_alpha": 2.0, "mg_fp32": 1},
    {"mg_tail_cells": 0},                       # every level grid-wide, coarsest smoothed
    {"mg_tail_cells": 0, "mg_fp32": 1},
    {"mg_tail_cells": 4000, "mg_fp32": 1},      # largest tail that fits the LDS
    {"mg_maxlevels": 3},                        # coarsest too large for the direct solve
    {"mg_maxlevels": 3, "mg_tail_cells": 4000, "mg_fp32": 1},
    {"mg_coarse_presweep": 1, "mg_coarse_postsweep": 1},
    {"mg_coarse_presweep": 0, "mg_coarse_postsweep": 2, "mg_fp32": 1},
    {"mg_presweep": 1, "mg_postsweep": 3},
    {"mg_smoother": 1},
    {"mg_smoother": 1, "mg_fp32": 1},
    {"mg_sell_rows": 1},                        # grid-wide coarse levels in sliced ELL
    {"mg_sell_rows": 1, "mg_fp32": 1},
    {"mg_sell_rows": 1, "mg_tail_cells": 0, "mg_fp32": 1},
    {"mg_sell_rows": 1, "mg_coarse_presweep": 0, "mg_coarse_postsweep": 2},
    {"mg_sell_rows": 0},                        # CSR on every coarse level
    {"mg_fuse_prolong": 0},                     # accepted, without effect
    {"mg_fuse_prolong": 0, "mg_fp32": 1, "mg_sell_rows": 1},
    {"mg_cycle": 1},                            # F cycle
    {"mg_cycle": 2, "mg_fp32": 1},              # W cycle
    {"mg_cycle": 2, "mg_tail_cells": 0, "mg_fp32": 1},
    {"mg_cycle": 1, "mg_sell_rows": 1, "mg_fuse_prolong": 0},
    {"mg_cycle": 2, "mg_smoother": 1},
]


def _ids(v):
    return ",".join(f"{k}={x}" for k, x in v.items()) or "default"


def _solve(nbr, nnbr, ac, anb, bc, solver, opts, lmg=2):
    m = fs.Mesh(nbr, nnbr)
    for k, v in opts.items():
        m.set_option(k, v)
    return m.solve_equation("pressc", np.zeros(len(ac)), 1e-8, 400, solver, lmg, ac, anb, bc)


@pytest.mark.parametrize("solver", ["bicgs", "cg", "gmres"])
@pytest.mark.parametrize("opts", VARIANTS, ids=_ids)
def test_neumann_variants_reach_1e8(neumann, solver, opts):
    asym = opts.get("mg_presweep", 2) != opts.get("mg_postsweep", 2) or \
        opts.get("mg_coarse_presweep", -1) != opts.get("mg_coarse_postsweep", -1)
    if solver == "cg" and (asym or opts.get("mg_cycle", 0)):
        pytest.skip("unequal pre/post sweeps, or the extra descents of F and W cycles, give a non-symmetric "
                    "cycle: not a CG preconditioner")
    nbr, nnbr, ac, anb, bc, A = neumann
    rc, fit, dphi, res4, st = _solve(nbr, nnbr, ac, anb, bc, solver, opts)
    assert rc == 0, st
    assert np.abs(bc - A @ dphi).sum() <= 1.0001e-8 * np.abs(bc).sum()
    # the cycle is a working preconditioner: far fewer iterations than unpreconditioned
    assert st["iterations"] < 60, st


@pytest.mark.parametrize("solver", ["bicgs", "cg", "gmres"])
@pytest.mark.parametrize("opts", [{}, {"mg_fp32": 1}, {"mg_tail_cells": 0}, {"mg_maxlevels": 3, "mg_fp32": 1},
                                  {"gmres_restart": 5}, {"mg_sell_rows": 1, "mg_fp32": 1},
                                  {"mg_sell_rows": 1, "mg_tail_cells": 0}],
                         ids=_ids)
def test_shifted_variants_match_direct(shifted, solver, opts):
    nbr, nnbr, ac, anb, bc, A, x = shifted
    rc, fit, dphi, res4, st = _solve(nbr, nnbr, ac, anb, bc, solver, opts)
    assert rc == 0, st
    assert np.abs(bc - A @ dphi).sum() <= 1.0001e-8 * np.abs(bc).sum()
    np.testing.assert_allclose(dphi, x, rtol=0, atol=1e-6 * np.abs(x).max())


@pytest.mark.parametrize("fp32", [0, 1])
def test_unfused_prolongation_is_bitwise_the_fused(neumann, fp32):
    """x + alpha*xc[parent] formed in the first post-sweep's loads or written
    by a pass of its own first: the same values in the same precision, so
    the same iterates."""
    nbr, nnbr, ac, anb, bc, A = neumann
    out = []
    for fuse in (1, 0):
        rc, fit, dphi, res4, st = _solve(nbr, nnbr, ac, anb, bc, "cg",
                                         {"mg_fp32": fp32, "mg_fuse_prolong": fuse, "mg_sell_rows": 1})
        assert rc == 0, st
        out.append((dphi, st["iterations"]))
    assert out[0][1] == out[1][1]
    assert np.array_equal(out[0][0], out[1][0])


def test_overcorrection_saves_iterations(neumann):
    """Scaling the injected coarse correction (alpha 1.7) needs fewer
    preconditioned iterations than the plain additive correction."""
    nbr, nnbr, ac, anb, bc, A = neumann
    its = {}
    for alpha in (1.0, 1.7):
        rc, fit, dphi, res4, st = _solve(nbr, nnbr, ac, anb, bc, "cg", {"mg_alpha": alpha, "mg_fp32": 1})
        assert rc == 0
        its[alpha] = st["iterations"]
    assert its[1.7] < its[1.0], its


@pytest.mark.parametrize("solver", ["cg", "gmres"])
def test_unpreconditioned_krylov(shifted, solver):
    nbr, nnbr, ac, anb, bc, A, x = shifted
    rc, fit, dphi, res4, st = _solve(nbr, nnbr, ac, anb, bc, solver, {"gmres_restart": 40}, lmg=0)
    assert rc == 0, st
    np.testing.assert_allclose(dphi, x, rtol=0, atol=1e-6 * np.abs(x).max())


def test_gmres_on_nonsymmetric_momentum_system():
    """GMRES + AMG on an upwind convection-diffusion (momentum-like) system."""
    nbr, nnbr, ac, anb, bc = systems.momentum_like(24, 20, 16, 5)
    A = systems.sparse(nbr, nnbr, ac, anb)
    x = spl.spsolve(A.tocsc(), bc)
    for fp32 in (0, 1):
        rc, fit, dphi, res4, st = _solve(nbr, nnbr, ac, anb, bc, "gmres", {"mg_fp32": fp32})
        assert rc == 0, st
        np.testing.assert_allclose(dphi, x, rtol=0, atol=1e-6 * np.abs(x).max())


def test_multigrid_as_solver_with_tail(shifted):
    """The reference's multigrid-as-solver loop (alpha 1) on the new cycle."""
    nbr, nnbr, ac, anb, bc, A, x = shifted
    its = {}
    for cyc in (0, 1, 2):
        for fp32 in (0, 1):
            m = fs.Mesh(nbr, nnbr)
            m.set_option("mg_fp32", fp32)
            m.set_option("mg_maxcycles", 300)
            m.set_option("mg_cycle", cyc)
            rc, fit, dphi, res4, st = m.solve_equation("pressc", np.zeros(len(ac)), 1e-8, 300, "sor", 1, ac, anb,
                                                       bc)
            assert rc == 0, st
            np.testing.assert_allclose(dphi, x, rtol=0, atol=1e-6 * np.abs(x).max())
            its[cyc, fp32] = st["iterations"]
    print("cycles to 1e-8 (V, F, W):", [its[c, 0] for c in (0, 1, 2)], flush=True)
    # the extra coarse-grid corrections of F and W cycles never cost cycles
    assert its[1, 0] <= its[0, 0] and its[2, 0] <= its[0, 0]


@pytest.mark.parametrize("alpha", [1.0, 1.3])
def test_cg_with_the_channel_f_cycle(neumann, alpha):
    """The channel's p' composition: CG preconditioned by the FP32 F-cycle with
    1/1 sweeps on every level and the coarse corrections over-relaxed.  The
    cycle is not symmetric, but CG's residual recurrence does not depend on
    the preconditioner, so a converged solve meets the stop rule on the true
    residual."""
    nbr, nnbr, ac, anb, bc, A = neumann
    opts = {"mg_cycle": 1, "mg_alpha": alpha, "mg_presweep": 1, "mg_postsweep": 1, "mg_coarse_presweep": 1,
            "mg_coarse_postsweep": 1, "mg_fp32": 1, "mg_fuse_prolong": 0}
    rc, fit, dphi, res4, st = _solve(nbr, nnbr, ac, anb, bc, "cg", opts)
    assert rc == 0, st
    assert np.abs(bc - A @ dphi).sum() <= 1.0001e-8 * np.abs(bc).sum()
    assert st["iterations"] < 60, st


def test_bad_cycle_rejected():
    nbr, nnbr, ac, anb, bc = systems.pressure_like(4, 4, 4, 1)
    m = fs.Mesh(nbr, nnbr)
    with pytest.raises(fs.FsError):
        m.set_option("mg_cycle", 3)


def test_bad_alpha_rejected():
    nbr, nnbr, ac, anb, bc = systems.pressure_like(4, 4, 4, 1)
    m = fs.Mesh(nbr, nnbr)
    with pytest.raises(fs.FsError):
        m.set_option("mg_alpha", 7.0)


def test_pbcg_with_amg_preconditioner(shifted):
    """PBCG with the V-cycle in place of its D-ILU asolve (for r and rr: the
    cycle is symmetric, as this operator is) reaches the stop rule and the
    direct solution; the reference's D-ILU PBCG is still far from it after
    the same iteration budget.  (The reference's minimum-residual shadow
    rr = A r keeps BiCG well behind BiCGSTAB or CG with the same cycle.)"""
    nbr, nnbr, ac, anb, bc, A, x = shifted
    rc, fit, dphi, res4, st = _solve(nbr, nnbr, ac, anb, bc, "pbcg", {}, lmg=2)
    assert rc == 0, st
    np.testing.assert_allclose(dphi, x, rtol=0, atol=1e-6 * np.abs(x).max())
    rc0, fit0, dphi0, res40, st0 = _solve(nbr, nnbr, ac, anb, bc, "pbcg", {}, lmg=0)
    assert rc0 == 1 and st0["final_l1"] > 1e3 * st["final_l1"], (st, st0)


def test_sliced_ell_cycle_matches_csr(neumann):
    """The sliced-ELL coarse levels change only the order of each row's sum:
    the same iteration count (within one) and the same solution."""
    nbr, nnbr, ac, anb, bc, A = neumann
    out = {}
    for rows in (0, 1):
        rc, fit, dphi, res4, st = _solve(nbr, nnbr, ac, anb, bc, "bicgs", {"mg_sell_rows": rows})
        assert rc == 0, st
        out[rows] = (st["iterations"], dphi - dphi.mean())
    assert abs(out[0][0] - out[1][0]) <= 1
    np.testing.assert_allclose(out[1][1], out[0][1], rtol=0, atol=1e-6 * np.abs(out[0][1]).max())
