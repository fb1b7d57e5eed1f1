"""Sensitivities (k_sens in csrc/tt_sens.inc) on grids whose blocks march several strands of layers side by side, against the
oracle: rods from 1 x 1 to 8 x 8 elements and sheets of few rows, with short and empty strands, for every objective; and
grids of one and two elements in x, whose tiles are 1 x 128 and 2 x 64 columns.

Tolerance: 1e-8, as in the other gradient tests (both sides solve to a relative residual of 1e-12 or better).
"""
import pytest

from oracle import oracle as O
from tests.gpu_helpers import problem, random_density, rel
from topopt_in_petsc_transient_amd import capi

pytestmark = pytest.mark.gpu

CASES = [((1, 1, 1030), o) for o in range(7)] + [((3, 3, 1100), o) for o in range(7)]
CASES += [(n, 3 + i % 4) for i, n in enumerate([(2, 2, 1537), (7, 7, 1030), (8, 8, 513), (5, 2, 1600), (40, 1, 300), (33, 2, 400),
                                               (65, 3, 350), (1, 129, 7), (1, 128, 3), (2, 65, 40), (2, 300, 120)])]


@pytest.mark.parametrize("nel,objective", CASES)
def test_sensitivities(nel, objective):
    print("sensitivities", nel, objective, flush=True)
    ex, ey, ez = nel
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
