"""Gradients on grids that take the column kernels (above 40,000 nodes, csrc/tt_apply_cols.inc), against the oracle: the
adjoint's split K / M product (two outputs, one staging buffer more, a second barrier per plane) and the objective's raw
products (no boundary mask) run there only, with the sensitivities and the Newmark right-hand side of the same grid.
Objectives 3, 4 and 6 use K alone, M alone and both; both boundary masks (the MBB beam's with its own load).  The grid is
ragged in every direction of the tiles.

The number of preconditioned iterations is held to that measured with these transfers and smoothers and a fifth more: a
flexible CG reaches the same states with a wrong correction from a coarser level, only later.

Tolerance: both sides solve to a relative residual of 1e-12 or better; 1e-8 is allowed for what the condition of the Newmark
operator and the steps make of it, as in the other gradient tests.
"""
import pytest

from oracle import oracle as O
from tests.gpu_helpers import problem, random_density, rel
from topopt_in_petsc_transient_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nel,nlvls", [((56, 32, 24), 3)])
@pytest.mark.parametrize("boundaries,loadloc", [(1, 2), (0, 0)])
@pytest.mark.parametrize("objective", [3, 4, 6])
def test_gradient_on_columns(nel, nlvls, boundaries, loadloc, objective):
    print("gradient", nel, boundaries, objective, flush=True)
    po, pg = problem(*nel, nsteps=3, dt=0.01, pulse_steps=2, objective=objective, nlvls=nlvls, boundaries=boundaries,
                     loadloc=loadloc)
    x = random_density(O.nel(po), seed=13)
    fx_ref, df_ref = O.objective_gradient(po, x, O.forward(po, x))
    assert fx_ref != 0.0
    c = capi.Context(pg)
    c.set_density(x)
    c.complete_initial_state()
    c.forward()
    fx, df = c.objective_gradient()
    c.close()
    assert abs(fx - fx_ref) <= 1e-8 * abs(fx_ref)
    assert rel(df, df_ref) < 1e-8


# (initial state and 4 steps: iterations in all)
@pytest.mark.parametrize("nel,nlvls,measured", [((24, 12, 12), 2, 54), ((24, 12, 12), 3, 51), ((16, 16, 16), 4, 50),
                                                ((20, 20, 20), 2, 54), ((12, 12, 12), 3, 57), ((56, 48, 48), 4, 84)])
@pytest.mark.parametrize("precision", [capi.TT_PREC_FP64, capi.TT_PREC_MIXED])
def test_iterations_of_the_preconditioned_solves(nel, nlvls, measured, precision):
    print("iterations", nel, nlvls, precision, flush=True)
    _, pg = problem(*nel, nsteps=4, dt=0.05, pulse_steps=3, nlvls=nlvls, precision=precision)
    c = capi.Context(pg)
    c.set_density(random_density(c.nel, seed=10))
    c.complete_initial_state()
    c.forward()
    iters = c.stats().krylov_iters
    c.close()
    assert iters <= 1.2 * measured
