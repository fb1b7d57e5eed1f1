"""Kernels at the edges of their tiles and of the rules that choose between them, against the oracle:

* sensitivities (csrc/tt_sens.inc): element grids on each tile width (4, 8, 16 and 32 columns), ragged in every
  direction, one element wide, and with several layers per part, for every objective;
* the filter's operator (32 x 8 node columns, parts of the planes): grids of one element, at and one past the tile edges;
* the V-cycle's prolongation through two, three and four levels, and the coarsest solve on both sides of the order up to
  which it is one dense product;
* the Gram-Schmidt of the basis solves through several groups of 8 vectors and a restart.

Tolerances: both sides solve to a relative residual of 1e-12 or better; the states, objective and gradient amplify it by
the condition of the Newmark operator and the number of steps, for which 1e-8 is allowed (1e-10 for one filter solve,
1e-9 for basis vectors).
"""
import numpy as np
import pytest

from oracle import oracle as O
from tests.gpu_helpers import problem, random_density, rel
from topopt_in_petsc_transient_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nel", [(1, 2, 3), (3, 65, 2), (8, 33, 4), (9, 16, 3), (17, 9, 2), (33, 8, 5), (3, 2, 700)])
@pytest.mark.parametrize("objective", range(7))
def test_sensitivities(nel, objective):
    ex, ey, ez = nel
    print("sensitivities", nel, objective, flush=True)
    po, pg = problem(*nel, nsteps=3, dt=0.002, pulse_steps=2, objective=objective, nlvls=1, lx=0.1 * ex, ly=0.1 * ey,
                     lz=0.1 * ez)
    x = random_density(O.nel(po), seed=8)
    fx_ref, df_ref = O.objective_gradient(po, x, O.forward(po, x))
    c = capi.Context(pg)
    c.set_density(x)
    c.complete_initial_state()
    c.forward()
    fx, df = c.objective_gradient()
    c.close()
    assert abs(fx - fx_ref) <= 1e-8 * abs(fx_ref)
    assert rel(df, df_ref) < 1e-8


@pytest.mark.parametrize("nel", [(1, 1, 1), (31, 7, 2), (32, 8, 1), (30, 6, 3), (2, 17, 40), (70, 3, 5), (3, 2, 300),
                                 (1, 20000, 1)])
def test_filter(nel):
    print("filter", nel, flush=True)
    po, pg = problem(*nel, nsteps=2, lx=0.05 * nel[0], ly=0.07 * nel[1], lz=0.04 * nel[2], nlvls=1, rmin=0.11)
    c = capi.Context(pg)
    x = random_density(c.nel, seed=9)
    out = c.pde_filter(x)
    c.close()
    assert rel(out, O.pde_filter(po, 0.11, x)) < 1e-10


# coarsest grids: 1,911, 336, 81, 3,993, 192 and 1,176 dofs; the last finest grid has 136,857 nodes (the wider prolongation)
@pytest.mark.parametrize("nel,nlvls", [((24, 12, 12), 2), ((24, 12, 12), 3), ((16, 16, 16), 4), ((20, 20, 20), 2),
                                       ((12, 12, 12), 3), ((56, 48, 48), 4)])
@pytest.mark.parametrize("precision", [capi.TT_PREC_FP64, capi.TT_PREC_MIXED])
def test_levels_and_coarsest_solve(nel, nlvls, precision):
    print("levels", nel, nlvls, precision, flush=True)
    po, pg = problem(*nel, nsteps=4, dt=0.05, pulse_steps=3, nlvls=nlvls, precision=precision)
    x = random_density(O.nel(po), seed=10)
    ref = O.forward(po, x)
    c = capi.Context(pg)
    c.set_density(x)
    c.complete_initial_state()
    c.forward()
    u, v, a = c.get_state(4)
    iters = c.stats().krylov_iters
    c.close()
    assert rel(u, ref[4, 0]) < 1e-8 and rel(v, ref[4, 1]) < 1e-8
    assert iters <= 5 * 40  # the preconditioner works at every depth


def test_long_thin_levels():
    """The coarser grid (1 x 1 x 9,500 elements) has more blocks and reduction partials than the finest."""
    po, pg = problem(2, 2, 19000, nsteps=2, dt=0.001, pulse_steps=2, nlvls=2, lx=0.2, ly=0.2, lz=1900.0)
    x = random_density(O.nel(po), seed=12)
    ref = O.forward(po, x)
    c = capi.Context(pg)
    c.set_density(x)
    c.complete_initial_state()
    c.forward()
    u, v, a = c.get_state(2)
    c.close()
    assert rel(u, ref[2, 0]) < 1e-8 and rel(v, ref[2, 1]) < 1e-8


def test_basis_solves_over_many_krylov_vectors():
    po, pg = problem(nelx=8, nely=4, nelz=4, nsteps=4, dt=0.05, pulse_steps=3, nlvls=1)
    pg.reduction, pg.basis, pg.omega0, pg.coarse_direct_max = 1, 3, 0.02, 1  # a weak preconditioner
    po.rtol = 1e-12
    x = random_density(O.nel(po), seed=11, lo=0.3)
    c = capi.Context(pg)
    c.set_density(x)
    c.complete_initial_state()
    c.forward()
    m = c.reduced_model(with_states=True)
    print("Krylov iterations", c.stats().krylov_iters, flush=True)
    c.close()
    ref = O.reduced_model(po, x, 3, 0.02)
    assert rel(m["Q"], ref["Q"]) < 1e-9
    assert np.allclose(m["Q"] @ m["Q"].T, np.eye(3), atol=1e-12)
