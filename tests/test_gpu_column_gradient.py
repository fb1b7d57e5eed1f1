"""Gradients on grids that take the column kernels (above 40,000 nodes, csrc/tt_apply_cols.inc), against the oracle: the
adjoint's split K / M product (two outputs, one staging buffer more, a second barrier per plane) and the objective's raw
products (no boundary mask) run there only, with the sensitivities and the Newmark right-hand side of the same grid.
Objectives 3, 4 and 6 use K alone, M alone and both; both boundary masks (the MBB beam's with its own load).  The grid is
ragged in every direction of the tiles.  The rods (few columns, many planes) cut a block's planes into strands that march side
by side; their last strands are short or empty.  Their single products go through the operator test's own check.

The number of preconditioned iterations is held to that measured with these transfers and smoothers and a fifth more: a
flexible CG reaches the same states with a wrong correction from a coarser level, only later.

Tolerance: both sides solve to a relative residual of 1e-12 or better; 1e-8 is allowed for what the condition of the Newmark
operator and the steps make of it, as in the other gradient tests.
"""
import pytest

from oracle import oracle as O
from tests.gpu_helpers import problem, random_density, rel
from tests.test_gpu_column_apply import test_column_apply_against_the_oracle as check_column_apply
from topopt_in_petsc_transient_amd import capi

pytestmark = pytest.mark.gpu


# rods: 21, 13, 8, 5, 3 and 2 strands in a block; the last grid's cross-section leaves no room for a second one
RODS = [(1, 1, 11111), (2, 2, 6000), (1, 7, 2600), (7, 1, 2700), (5, 5, 1200), (7, 7, 701), (9, 9, 444), (2, 20, 700),
        (10, 10, 400)]


@pytest.mark.parametrize("nel", RODS)
@pytest.mark.parametrize("boundaries", [0, 1])
def test_rod_apply_against_the_oracle(nel, boundaries):
    print("rod", nel, boundaries, flush=True)
    check_column_apply(nel, boundaries)


@pytest.mark.parametrize("nel,nlvls", [((56, 32, 24), 3), ((2, 2, 6000), 2), ((7, 7, 701), 1)])
@pytest.mark.parametrize("boundaries,loadloc", [(1, 2), (0, 0)])
@pytest.mark.parametrize("objective", [3, 4, 6])
def test_gradient_on_columns(nel, nlvls, boundaries, loadloc, objective):
    print("gradient", nel, boundaries, objective, flush=True)
    lengths = {} if nel[2] < 100 else dict(zip(("lx", "ly", "lz"), (0.05 * e for e in nel)))
    po, pg = problem(*nel, nsteps=3, dt=0.01, pulse_steps=2, objective=objective, nlvls=nlvls, boundaries=boundaries,
                     loadloc=loadloc, **lengths)
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
