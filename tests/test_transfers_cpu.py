"""The multigrid transfers (k_restrict, k_prolong_chain in csrc/tt_kernels.hip), their source compiled for the CPU and run
thread by thread, against plain 1-D interpolation matrices:

* prolongation: the one-pass sum over all coarser levels equals the nested masked prolongations, level by level, that it
  stands for (x_l += P x_{l+1} on free dofs, then the next finer level), for both boundary masks, one to three coarser
  levels, either number of planes per thread, FP64, FP32 and FP32 with an FP64 coarsest vector; dofs clamped on the fine
  level keep their bits;
* restriction: the transpose of the prolongation, 0 on clamped coarse dofs, with a node or a dof per thread.

Tolerances, from the operation counts: a dof of the prolongation sums 8 weighted values per level (at most 3 levels, about
20 rounded operations each) and one of the restriction 27, so 64 eps relative to the norm in either precision.
"""
import ctypes
import os
import re
import subprocess

import numpy as np
import pytest
import scipy.sparse as sp

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "topopt_in_petsc_transient_amd", "csrc")

SHIM = r"""
#include <cmath>
#include <cstddef>
#include <cstdint>
using std::fma;
#define __global__ static
#define __device__ static
#define __host__
#define __forceinline__ inline
struct Dim { unsigned x; };
static Dim blockIdx, blockDim, threadIdx;
struct GridArgs { int nx, ny, nz, ex, ey, ez; };
"""
CALLS = r"""
template <class F> static void each_thread(long n, unsigned bs, F f) {
    blockDim.x = bs;
    for (long b = 0; b * bs < n; b++)
        for (unsigned t = 0; t < bs; t++) { blockIdx.x = (unsigned)b; threadIdx.x = t; f(); }
}
static GridArgs grid(const int* n) { return GridArgs{n[0], n[1], n[2], n[0] - 1, n[1] - 1, n[2] - 1}; }
template <int NZ, typename Tf, typename Tl>
static void prolong(const int* n, int levels, void* const* x, const uint8_t* mask, void* xf) {
    ProlongChain pc{};
    pc.n = levels;
    for (int l = 0; l < levels; l++) {
        pc.x[l] = x[l];
        pc.nx[l] = n[3 * (l + 1)]; pc.ny[l] = n[3 * (l + 1) + 1]; pc.nz[l] = n[3 * (l + 1) + 2];
    }
    const GridArgs f = grid(n);
    each_thread((long)f.nx * ((f.ny + 1) / 2) * ((f.nz + NZ - 1) / NZ), 64,
                [&] { k_prolong_chain<NZ, Tf, Tl>(f, pc, mask, (Tf*)xf); });
}
template <int NC, typename Tf, typename Tc>
static void restrict_(const int* n, const void* rf, const uint8_t* cmask, void* bc) {
    const GridArgs f = grid(n), c = grid(n + 3);
    each_thread((long)c.nx * c.ny * c.nz * (3 / NC), NC == 3 ? 64 : 128,
                [&] { k_restrict<NC, Tf, Tc>(f, c, (const Tf*)rf, cmask, (Tc*)bc); });
}
// types: 0 FP64, 1 FP32 fine with an FP64 coarsest / coarse vector, 2 FP32
extern "C" void run_prolong(const int* n, int levels, void* const* x, const uint8_t* mask, void* xf, int types, int nz) {
    if (types == 0) nz == 2 ? prolong<2, double, double>(n, levels, x, mask, xf) : prolong<1, double, double>(n, levels, x, mask, xf);
    if (types == 1) nz == 2 ? prolong<2, float, double>(n, levels, x, mask, xf) : prolong<1, float, double>(n, levels, x, mask, xf);
    if (types == 2) nz == 2 ? prolong<2, float, float>(n, levels, x, mask, xf) : prolong<1, float, float>(n, levels, x, mask, xf);
}
extern "C" void run_restrict(const int* n, const void* rf, const uint8_t* cmask, void* bc, int types, int nc) {
    if (types == 0) nc == 3 ? restrict_<3, double, double>(n, rf, cmask, bc) : restrict_<1, double, double>(n, rf, cmask, bc);
    if (types == 1) nc == 3 ? restrict_<3, float, double>(n, rf, cmask, bc) : restrict_<1, float, double>(n, rf, cmask, bc);
    if (types == 2) nc == 3 ? restrict_<3, float, float>(n, rf, cmask, bc) : restrict_<1, float, float>(n, rf, cmask, bc);
}
"""


def _between(text, first, last):
    m = re.search(re.escape(first) + r".*?(?=" + re.escape(last) + ")", text, re.S)
    assert m, (first, last)
    return m.group(0)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    kernels = open(os.path.join(CSRC, "tt_kernels.hip")).read()
    header = open(os.path.join(CSRC, "tt_internal.h")).read()
    src = (SHIM + _between(header, "__host__ __device__ inline void grid_ijk", "//")
           + _between(kernels, "template <int NC, typename Tf, typename Tc>\n__global__ void k_restrict",
                      "void launch_restrict")
           + _between(kernels, "struct ProlongChain {", "void launch_prolong_chain") + CALLS)
    d = tmp_path_factory.mktemp("transfers")
    (d / "transfers.cpp").write_text(src)
    so = str(d / "transfers.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wno-unknown-pragmas", str(d / "transfers.cpp"),
                    "-o", so], check=True, capture_output=True)
    return ctypes.CDLL(so)


def _levels(nel, n):
    return [tuple(e >> l for e in nel) for l in range(n)]


def _mask(nel, boundaries):
    """Clamped dofs of a level (nz, ny, nx bits): the cantilever's face, or the MBB beam's face and edge."""
    m = np.zeros((nel[2] + 1, nel[1] + 1, nel[0] + 1), np.uint8)
    m[:, :, 0] = 7 if boundaries == 1 else 3
    if boundaries == 0:
        m[0, :, -1] |= 6
    return m.ravel()


def _clamped(m):
    return ((m[:, None] >> np.arange(3)) & 1).astype(bool).ravel()


def _p1(e):
    """Linear interpolation from e / 2 elements to e."""
    p = np.zeros((e + 1, e // 2 + 1))
    for i in range(e + 1):
        p[i, i // 2] += 0.5
        p[i, (i + 1) // 2] += 0.5
    return sp.csr_matrix(p)


def _p(nel):
    x, y, z = (_p1(e) for e in nel)
    return sp.kron(sp.kron(sp.kron(z, y), x), sp.identity(3)).tocsr()


GRIDS = [((2, 2, 2), 2), ((6, 2, 4), 2), ((2, 10, 6), 2), ((8, 4, 4), 3), ((4, 12, 8), 3), ((8, 16, 8), 4), ((24, 8, 16), 4)]
TYPES = {0: (np.float64, np.float64, 2.0 ** -52), 1: (np.float32, np.float64, 2.0 ** -23),
         2: (np.float32, np.float32, 2.0 ** -23)}  # fine, last coarse, eps


def _dims(lv):
    return (ctypes.c_int * (3 * len(lv)))(*[e + 1 for nel in lv for e in nel])


@pytest.mark.parametrize("nel,nlvls", GRIDS)
@pytest.mark.parametrize("boundaries", [0, 1])
@pytest.mark.parametrize("types", [0, 1, 2])
@pytest.mark.parametrize("nz", [1, 2])
def test_prolongation_through_all_levels(lib, nel, nlvls, boundaries, types, nz):
    tf, tl, eps = TYPES[types]
    lv = _levels(nel, nlvls)
    rng = np.random.default_rng(1)
    x = []
    for l, e in enumerate(lv):
        v = rng.standard_normal(3 * np.prod([q + 1 for q in e])).astype(tl if l == nlvls - 1 else tf)
        if l:
            v[_clamped(_mask(e, boundaries))] = 0.0  # a level's correction is 0 there
        x.append(v)
    ref = [v.astype(np.float64) for v in x]
    for l in range(nlvls - 2, -1, -1):
        free = ~_clamped(_mask(lv[l], boundaries))
        ref[l][free] += (_p(lv[l]) @ ref[l + 1])[free]
    got = x[0].copy()
    ptrs = (ctypes.c_void_p * (nlvls - 1))(*[v.ctypes.data for v in x[1:]])
    m = _mask(nel, boundaries)
    lib.run_prolong(_dims(lv), nlvls - 1, ptrs, m.ctypes.data_as(ctypes.c_void_p), got.ctypes.data_as(ctypes.c_void_p),
                    types, nz)
    assert np.linalg.norm(got - ref[0]) <= 64 * eps * np.linalg.norm(ref[0])
    cl = _clamped(m)
    assert np.array_equal(got[cl], x[0][cl])


@pytest.mark.parametrize("nel", [g[0] for g in GRIDS])
@pytest.mark.parametrize("boundaries", [0, 1])
@pytest.mark.parametrize("types", [0, 1, 2])
@pytest.mark.parametrize("nc", [1, 3])
def test_restriction_is_the_transpose(lib, nel, boundaries, types, nc):
    tf, tc, eps = TYPES[types]
    lv = _levels(nel, 2)
    r = np.random.default_rng(2).standard_normal(3 * np.prod([q + 1 for q in nel])).astype(tf)
    m = _mask(lv[1], boundaries)
    ref = _p(nel).T @ r.astype(np.float64)
    ref[_clamped(m)] = 0.0
    got = np.full(ref.size, np.nan, tc)
    lib.run_restrict(_dims(lv), r.ctypes.data_as(ctypes.c_void_p), m.ctypes.data_as(ctypes.c_void_p),
                     got.ctypes.data_as(ctypes.c_void_p), types, nc)
    assert np.linalg.norm(got - ref) <= 64 * eps * np.linalg.norm(ref)
    assert not got[_clamped(m)].any()
