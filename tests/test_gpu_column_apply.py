"""The operator kernels (csrc/tt_apply_box.inc for small grids, csrc/tt_apply_cols.inc for the others) against the oracle
where their tilings can go wrong: grids of one element, single rows and planes, extents at and around the tile edges,
long thin boxes, the sizes on both sides of the rule between the two kernels, with both boundary masks (clamped dofs
inside and at the edges of tiles).

Tolerance: a result is a sum of at most 8 element contributions, each reached through about 25 rounded operations from
the inputs (3 + 3 levels of sums, the block products, the coefficients), and the element products of random inputs do
not cancel: 32 eps relative to the norm, in FP64 twice that for the oracle's own rounding.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.gpu_helpers import problem, random_density, rel
from topopt_in_petsc_transient_amd import capi

pytestmark = pytest.mark.gpu

GRIDS = [(1, 1, 1), (2, 1, 3), (7, 5, 3), (15, 15, 2), (16, 8, 9), (17, 31, 1), (3, 70, 2), (130, 2, 2), (2, 3, 150),
         (61, 43, 5),
         # above 40,000 nodes: the column kernel
         (130, 20, 15), (17, 47, 50), (300, 11, 12), (3, 3, 3000), (2, 4000, 3), (3999, 2, 3), (31, 31, 39), (15, 49, 49)]


@pytest.mark.parametrize("nel", GRIDS)
@pytest.mark.parametrize("boundaries", [0, 1])
def test_column_apply_against_the_oracle(nel, boundaries):
    po, pg = problem(*nel, nsteps=2, lx=1.3, ly=0.7, lz=2.1, nlvls=1, boundaries=boundaries)
    pg.coarse_direct_max = 1  # (no dense inverse: the operator alone is tested)
    c = capi.Context(pg)
    x = random_density(c.nel, 3)
    c.set_density(x)
    u = np.random.default_rng(5).standard_normal(c.nd).astype(np.float32).astype(np.float64)
    N = O.bc_mask(po)
    a = O.newmark_consts(1, po.t1 / po.nsteps)
    u64 = torch.from_numpy(u).cuda()
    u32 = u64.float()
    y64, y32 = torch.empty_like(u64), torch.empty_like(u32)
    torch.cuda.synchronize()
    for which, cK, cM in ((capi.TT_OP_K, 1.0, 0.0), (capi.TT_OP_M, 0.0, 1.0),
                          (capi.TT_OP_A, 1.0 + a[2] * po.dbeta, a[5] + a[2] * po.dalpha)):
        ref = O.apply_bc(po, x, cK, cM, u, N)
        c.op_apply(which, u64, y64, prec=0)
        c.op_apply(which, u32, y32, prec=1)
        assert rel(y64.cpu().numpy(), ref) < 64 * 2.2e-16, (which, "FP64")
        assert rel(y32.double().cpu().numpy(), ref) < 32 * 6e-8, (which, "FP32")
    c.close()
