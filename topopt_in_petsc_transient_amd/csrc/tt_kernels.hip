// HIP kernels for gfx950: matrix-free SIMP hex8 operator, multigrid transfers,
// Krylov vector kernels and deterministic reductions.
//
// The operator y = sum_e (cK*kfac_e*KE + cM*mfac_e*ME) u_e of the reference's
// assembled AIJ matrices (LinearElasticity.cc:2502-2619) is applied element by
// element in the element's symmetry-adapted basis (tt_apply_cols.inc; small
// grids tt_apply_box.inc), with the corner values added per node in a fixed
// order: no atomics, results are bit-reproducible.  Epilogue functors fuse the
// Krylov / Chebyshev vector work into the same pass.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "tt_internal.h"

namespace tt {

// ------------------------------------------------------------------ helpers
// Element i of p through a 32-bit byte offset from a uniform base (scalar-base addressing; every
// array here is below 4 GiB, which the context checks at creation).
template <typename T>
__device__ __forceinline__ T ld(const T* p, unsigned i) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + i * (unsigned)sizeof(T));
}
__device__ __forceinline__ double coef_ld(const double* p, long i) { return p[i]; }
__device__ __forceinline__ double coef_ld(const float* p, long i) { return (double)p[i]; }
__device__ __forceinline__ double coef_ld(const bf16_t* p, long i) {
    return (double)__uint_as_float(((uint32_t)p[i]) << 16);
}

// A uniform pointer as a scalar base in global memory: what is added to it per lane stays a 32-bit byte offset (the
// compiler would otherwise hoist base + lane offset out of a loop over planes into 64-bit vector address pairs).
template <typename T>
using gptr = __attribute__((address_space(1))) T*;
template <typename T>
__device__ __forceinline__ gptr<T> sbase(T* p) {
    gptr<T> g = (gptr<T>)p;
    asm("" : "+s"(g));
    return g;
}
// A lane's offset as byte offsets of 1, 2, 4 and 8 byte elements, opaque to the compiler (it would widen the scaling to
// 64 bits); what a kernel does not use costs nothing.
struct LaneOff {
    unsigned o1, o2, o4, o8;
    __device__ __forceinline__ explicit LaneOff(unsigned i = 0) : o1(i), o2(2 * i), o4(4 * i), o8(8 * i) {
        asm("" : "+v"(o1));
        asm("" : "+v"(o2));
        asm("" : "+v"(o4));
        asm("" : "+v"(o8));
    }
    template <typename T>
    __device__ __forceinline__ unsigned of() const {
        return sizeof(T) == 1 ? o1 : sizeof(T) == 2 ? o2 : sizeof(T) == 4 ? o4 : o8;
    }
};
// element i (+ c, an immediate) of a uniform pointer
template <typename T>
__device__ __forceinline__ T ldu(const T* p, const LaneOff& i, int c = 0) {
    typedef __attribute__((address_space(1))) const char* cp;
    return ((gptr<const T>)((cp)sbase(p) + i.of<T>()))[c];
}
// The three consecutive values of one node at dofs b + i .. b + i + 2 (b uniform, i per lane).
template <typename T>
__device__ __forceinline__ void ld3(const T* p, size_t b, const LaneOff& i, T (&v)[3]) {
    typedef __attribute__((address_space(1))) const char* cp;
    const gptr<const T> q = (gptr<const T>)((cp)sbase(p + b) + i.of<T>());
#pragma unroll
    for (int c = 0; c < 3; c++) v[c] = q[c];
}
template <typename T>
__device__ __forceinline__ void st3(T* p, size_t b, const LaneOff& i, const T (&v)[3]) {
    typedef __attribute__((address_space(1))) char* cp;
    const gptr<T> q = (gptr<T>)((cp)sbase(p + b) + i.of<T>());
#pragma unroll
    for (int c = 0; c < 3; c++) q[c] = v[c];
}
__device__ __forceinline__ double coef_val(double v) { return v; }
__device__ __forceinline__ float coef_val(float v) { return v; }
__device__ __forceinline__ float coef_val(bf16_t v) { return __uint_as_float((uint32_t)v << 16); }

constexpr int BS = 256;  // threads per block for all 1-D kernels

// ------------------------------------------------------------------ deterministic block reduction
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV], double* sh) {
    // sh: BS/64 * NV doubles
#pragma unroll
    for (int k = 0; k < NV; k++) {
        double x = v[k];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
        v[k] = x;
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < NV; k++) sh[wid * NV + k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < NV; k++) {
            double s = 0.0;
            for (int w = 0; w < (int)(blockDim.x >> 6); w++) s += sh[w * NV + k];
            v[k] = s;
        }
    }
}

// Writes the block's NV partial sums to part[block*NV + k] (plain stores).
template <int NV>
__device__ __forceinline__ void write_partials(double (&v)[NV], double* part) {
    __shared__ double sh[16 * NV];
    block_sum<NV>(v, sh);
    if (threadIdx.x == 0) {
        const unsigned bid = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
#pragma unroll
        for (int k = 0; k < NV; k++) part[(size_t)bid * NV + k] = v[k];
    }
}

// Sum of partials written by an earlier kernel; every thread of the block gets the totals.
// Thread t sums blocks t, t + blockDim, ... (a fixed order for a given block size), then the
// waves are combined by a fixed butterfly and a fixed wave order, so every block of a launch
// obtains bit-identical totals.
template <int NV>
__device__ __forceinline__ void sum_partials(const double* __restrict__ part, int nblk, double (&out)[NV]) {
    __shared__ double sh[16 * NV];
    // four independent accumulators per thread so that four loads are in flight; fixed order
    double acc[NV], a4[3][NV];
#pragma unroll
    for (int k = 0; k < NV; k++) acc[k] = a4[0][k] = a4[1][k] = a4[2][k] = 0.0;
    const int st = blockDim.x;
    int b = threadIdx.x;
    for (; b + 3 * st < nblk; b += 4 * st)
#pragma unroll
        for (int k = 0; k < NV; k++) {
            acc[k] += part[(size_t)b * NV + k];
            a4[0][k] += part[(size_t)(b + st) * NV + k];
            a4[1][k] += part[(size_t)(b + 2 * st) * NV + k];
            a4[2][k] += part[(size_t)(b + 3 * st) * NV + k];
        }
    for (; b < nblk; b += st)
#pragma unroll
        for (int k = 0; k < NV; k++) acc[k] += part[(size_t)b * NV + k];
#pragma unroll
    for (int k = 0; k < NV; k++) acc[k] += (a4[0][k] + a4[1][k]) + a4[2][k];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (int)(blockDim.x + 63) >> 6;
#pragma unroll
    for (int k = 0; k < NV; k++) {
        double x = acc[k];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
        if (lane == 0) sh[wid * NV + k] = x;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; k++) {
        double x = 0.0;
        for (int w = 0; w < nw; w++) x += sh[w * NV + k];
        out[k] = x;
    }
    __syncthreads();  // sh may be reused by a later call in the same kernel
}

void Reducer::init(int maxb) {
    maxblocks = maxb;
    partials.alloc((size_t)PB_COUNT * maxb * 4);
    scal.alloc(SC_COUNT);
    TT_HIP(hipMemset(partials.p, 0, sizeof(double) * PB_COUNT * maxb * 4));
    TT_HIP(hipMemset(scal.p, 0, sizeof(double) * SC_COUNT));
    TT_HIP(hipHostMalloc((void**)&host, sizeof(double) * SC_COUNT, hipHostMallocDefault));
    TT_HIP(hipHostMalloc((void**)&hpart, sizeof(double) * maxb * 4, hipHostMallocDefault));
    TT_HIP(hipHostMalloc((void**)&look, sizeof(double) * (kLookBB + 1), hipHostMallocMapped | hipHostMallocCoherent));
    TT_HIP(hipHostGetDevicePointer((void**)&look_dev, look, 0));
    for (int i = 0; i <= kLookBB; i++) look[i] = 0.0;
}
void Reducer::host_sum(int region, hipStream_t s, double* out) {
    const int nb = nblk[region], v = nv[region];
    TT_HIP(hipMemcpyAsync(hpart, part(region), sizeof(double) * nb * v, hipMemcpyDeviceToHost, s));
    TT_HIP(hipStreamSynchronize(s));
    for (int k = 0; k < v; k++) out[k] = 0.0;
    for (int b = 0; b < nb; b++)
        for (int k = 0; k < v; k++) out[k] += hpart[(size_t)b * v + k];
}
Reducer::~Reducer() {
    if (host) (void)hipHostFree(host);
    if (hpart) (void)hipHostFree(hpart);
    if (look) (void)hipHostFree(look);
}

static inline int nblocks(long n, int per = BS) { return (int)((n + per - 1) / per); }
static inline int red_blocks(long n) {
    int b = nblocks(n);
    return b > 2048 ? 2048 : (b < 1 ? 1 : b);
}

// ------------------------------------------------------------------ operator apply
struct GridArgs {
    int nx, ny, nz, ex, ey, ez;
};
static inline GridArgs gargs(const Grid& g) { return GridArgs{g.nx, g.ny, g.nz, g.ex, g.ey, g.ez}; }

// Input staging policies of the column kernels: raw() loads what the staged value of a dof (at b + i + c, b uniform) is
// made of, value() makes it (two values where K and M act on different vectors).  depth: planes the loads run ahead (the
// three-vector form holds too much in flight for two).
template <typename T>
struct StageOne {  // w = u
    static constexpr int inputs = 1, depth = 2;
    const T* u;
    typedef T Raw;
    __device__ __forceinline__ Raw raw(size_t b, const LaneOff& i, int c = 0) const { return ldu(u + b, i, c); }
    __device__ __forceinline__ void value(const Raw& r, T (&x)[1]) const { x[0] = r; }
};
// First Chebyshev iterate x0 = c1 D^-1 b formed on the fly, with b = (T) r (FP64) on the finest level
template <typename T, bool FROM64>
struct StageChebFirst {
    static constexpr int inputs = 1, depth = 2;
    const double* r64;
    const T* b;
    const T* dinv;
    T c1;
    struct Raw {
        typename std::conditional<FROM64, double, T>::type b;
        T di;
    };
    __device__ __forceinline__ Raw raw(size_t base, const LaneOff& i, int c = 0) const {
        Raw r;
        if constexpr (FROM64) r.b = ldu(r64 + base, i, c);
        else r.b = ldu(b + base, i, c);
        r.di = ldu(dinv + base, i, c);
        return r;
    }
    __device__ __forceinline__ void value(const Raw& r, T (&x)[1]) const { x[0] = c1 * r.di * (T)r.b; }
};
struct StageThree {  // wK = sum_i cK_i in_i, wM = sum_i cM_i in_i (FP64)
    static constexpr int inputs = 2, depth = 1;
    const double *u, *v, *a;
    double k0, k1, k2, m0, m1, m2;
    struct Raw {
        double u, v, a;
    };
    __device__ __forceinline__ Raw raw(size_t b, const LaneOff& i, int c = 0) const {
        return Raw{ldu(u + b, i, c), ldu(v + b, i, c), ldu(a + b, i, c)};
    }
    __device__ __forceinline__ void value(const Raw& r, double (&x)[2]) const {
        x[0] = k0 * r.u + k1 * r.v + k2 * r.a;
        x[1] = m0 * r.u + m1 * r.v + m2 * r.a;
    }
};

#include "tt_apply_cols.inc"
#include "tt_apply_box.inc"
#include "tt_sens.inc"

// ---- epilogues.  A node's three dofs are b + i .. b + i + 2, b uniform over the block (its node plane's first dof, or
// 0).  fetch() loads the per-node operands an epilogue reads (its Pre) for one owned node, ahead of the element
// contraction.  put() then handles that node (inside the grid): cl are its clamped dofs, uo its input values (not
// masked); it may add to the thread's reduction share.  prologue() runs before the first put(), on every thread of a block
// that has a tile (block 0 always has one).  done() is called once by every thread of the block at the end (reducing
// epilogues write their block partial there).
// outputs: 2 where K and M results are taken apart (yK, yM), else yK is their sum; uses_input: whether put() reads uo.
#define TT_NO_PRE                                                     \
    struct Pre {};                                                    \
    template <class S>                                                \
    __device__ __forceinline__ void fetch(size_t, const LaneOff&, const S&, Pre&) const {}

template <typename T>
struct EpiBC {  // y = A u on free dofs, u on clamped
    static constexpr int outputs = 1;
    static constexpr bool uses_input = true;
    T* y;
    TT_NO_PRE
    __device__ void put(size_t b, const LaneOff& i, uint8_t cl, const T (&yK)[3], const T (&)[3], const T (&uo)[3],
                        double (&)[2], const Pre&) const {
        T v[3];
#pragma unroll
        for (int c = 0; c < 3; c++) v[c] = ((cl >> c) & 1) ? uo[c] : yK[c];
        st3(y, b, i, v);
    }
    __device__ void prologue() {}
    __device__ void done(double (&)[2]) const {}
};

template <typename T>
struct EpiBCDot {  // y = A u (BC form) and partials of u.y
    static constexpr int outputs = 1;
    static constexpr bool uses_input = true;
    T* y;
    double* part;
    TT_NO_PRE
    __device__ void put(size_t b, const LaneOff& i, uint8_t cl, const T (&yK)[3], const T (&)[3], const T (&uo)[3],
                        double (&acc)[2], const Pre&) const {
        T v[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            v[c] = ((cl >> c) & 1) ? uo[c] : yK[c];
            acc[0] += (double)uo[c] * (double)v[c];
        }
        st3(y, b, i, v);
    }
    __device__ void prologue() {}
    __device__ void done(double (&acc)[2]) const {
        double a[1] = {acc[0]};
        write_partials<1>(a, part);
    }
};

template <typename T>
struct EpiResid {  // r = b - A x
    static constexpr int outputs = 1;
    static constexpr bool uses_input = true;
    const T* rhs;
    T* r;
    struct Pre {
        T b[3];
    };
    template <class S>
    __device__ __forceinline__ void fetch(size_t b, const LaneOff& i, const S&, Pre& p) const { ld3(rhs, b, i, p.b); }
    __device__ void put(size_t b, const LaneOff& i, uint8_t cl, const T (&yK)[3], const T (&)[3], const T (&uo)[3],
                        double (&)[2], const Pre& p) const {
        T v[3];
#pragma unroll
        for (int c = 0; c < 3; c++) v[c] = p.b[c] - (((cl >> c) & 1) ? uo[c] : yK[c]);
        st3(r, b, i, v);
    }
    __device__ void prologue() {}
    __device__ void done(double (&)[2]) const {}
};

// One damped-Jacobi step from x = 0 and its residual in one pass (an intermediate multigrid level's
// pre-smoothing): x = c1 D^-1 b is formed in staging (StageChebFirst) and written, with r = b - A x.
template <typename T>
struct EpiResidFirst {
    static constexpr int outputs = 1;
    static constexpr bool uses_input = true;
    T* x;
    T* r;
    struct Pre {
        T b[3];
    };
    template <class S>
    __device__ __forceinline__ void fetch(size_t b, const LaneOff& i, const S& st, Pre& p) const { ld3(st.b, b, i, p.b); }
    __device__ void put(size_t b, const LaneOff& i, uint8_t cl, const T (&yK)[3], const T (&)[3], const T (&uo)[3],
                        double (&)[2], const Pre& p) const {
        T v[3];
#pragma unroll
        for (int c = 0; c < 3; c++) v[c] = p.b[c] - (((cl >> c) & 1) ? uo[c] : yK[c]);
        st3(x, b, i, uo);
        st3(r, b, i, v);
    }
    __device__ void prologue() {}
    __device__ void done(double (&)[2]) const {}
};

// r = b - A x (FP64) with the partials of b.b and r.r, one per block into each of two regions
struct EpiResidDots {
    static constexpr int outputs = 1;
    static constexpr bool uses_input = true;
    const double* rhs;
    double* r;
    double* pbb;
    double* prr;
    struct Pre {
        double b[3];
    };
    template <class S>
    __device__ __forceinline__ void fetch(size_t b, const LaneOff& i, const S&, Pre& p) const { ld3(rhs, b, i, p.b); }
    __device__ void put(size_t b, const LaneOff& i, uint8_t cl, const double (&yK)[3], const double (&)[3],
                        const double (&uo)[3], double (&acc)[2], const Pre& p) const {
        double v[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            v[c] = p.b[c] - (((cl >> c) & 1) ? uo[c] : yK[c]);
            acc[0] = fma(p.b[c], p.b[c], acc[0]);
            acc[1] = fma(v[c], v[c], acc[1]);
        }
        st3(r, b, i, v);
    }
    __device__ void prologue() {}
    __device__ void done(double (&acc)[2]) const {
        __shared__ double sh[16 * 2];
        block_sum<2>(acc, sh);
        if (threadIdx.x == 0) {
            const unsigned bid = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
            pbb[bid] = acc[0];
            prr[bid] = acc[1];
        }
    }
};

template <typename T>
struct EpiCheb {  // r = b - A x; dn = c0 d + c1 dinv r; xn = x + dn
    static constexpr int outputs = 1;
    static constexpr bool uses_input = true;
    const T* rhs;
    const T* d;
    const T* dinv;
    T c0, c1;
    T* xn;
    T* dn;
    struct Pre {
        T b[3], d[3], di[3];
    };
    template <class S>
    __device__ __forceinline__ void fetch(size_t b, const LaneOff& i, const S&, Pre& p) const {
        ld3(rhs, b, i, p.b);
        ld3(dinv, b, i, p.di);
        if (d) ld3(d, b, i, p.d);
    }
    __device__ void put(size_t b, const LaneOff& i, uint8_t cl, const T (&yK)[3], const T (&)[3], const T (&uo)[3],
                        double (&)[2], const Pre& p) const {
        T dd[3], v[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const T r = p.b[c] - (((cl >> c) & 1) ? uo[c] : yK[c]);
            dd[c] = c1 * p.di[c] * r;
            if (d) dd[c] = fma(c0, p.d[c], dd[c]);
            v[c] = uo[c] + dd[c];
        }
        st3(xn, b, i, v);
        if (dn) st3(dn, b, i, dd);
    }
    __device__ void prologue() {}
    __device__ void done(double (&)[2]) const {}
};

// Second Chebyshev step from x0 = c1 D^-1 b (staged by StageChebFirst, so d = x0):
// dn = c0 x0 + c1 D^-1 (b - A x0), xn = x0 + dn; on the finest level it also writes b = (T) r.
template <typename T, bool FROM64>
struct EpiChebFirst {
    static constexpr int outputs = 1;
    static constexpr bool uses_input = true;
    T* bout;
    const T* dinv;
    T c0, c1;
    T* xn;
    T* dn;
    struct Pre {
        typename std::conditional<FROM64, double, T>::type b[3];
        T di[3];
    };
    template <class S>
    __device__ __forceinline__ void fetch(size_t b, const LaneOff& i, const S& st, Pre& p) const {
        if constexpr (FROM64) ld3(st.r64, b, i, p.b);
        else ld3(st.b, b, i, p.b);
        ld3(dinv, b, i, p.di);
    }
    __device__ void put(size_t b, const LaneOff& i, uint8_t cl, const T (&yK)[3], const T (&)[3], const T (&uo)[3],
                        double (&)[2], const Pre& p) const {
        T bi[3], dd[3], v[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            bi[c] = (T)p.b[c];
            const T ax = ((cl >> c) & 1) ? uo[c] : yK[c];
            dd[c] = fma(c0, uo[c], c1 * p.di[c] * (bi[c] - ax));
            v[c] = uo[c] + dd[c];
        }
        if (FROM64) st3(bout, b, i, bi);
        st3(xn, b, i, v);
        st3(dn, b, i, dd);
    }
    __device__ void prologue() {}
    __device__ void done(double (&)[2]) const {}
};

// Last post-smoothing step of the finest level: z = x + c0 d + c1 D^-1 (b - A x) written in FP64
// as the preconditioned residual of flexible CG, with partials of z.r and z.q_old.
template <typename T>
struct EpiChebOut {
    static constexpr int outputs = 1;
    static constexpr bool uses_input = true;
    const T* rhs;
    const T* d;
    const T* dinv;
    T c0, c1;
    double* z;
    const double* r;
    const double* q;
    int first;
    double* part;
    struct Pre {
        T b[3], d[3], di[3];
        double r[3], q[3];
    };
    template <class S>
    __device__ __forceinline__ void fetch(size_t b, const LaneOff& i, const S&, Pre& p) const {
        ld3(rhs, b, i, p.b);
        ld3(dinv, b, i, p.di);
        if (d) ld3(d, b, i, p.d);
        ld3(r, b, i, p.r);
        if (!first) ld3(q, b, i, p.q);
    }
    __device__ void put(size_t b, const LaneOff& i, uint8_t cl, const T (&yK)[3], const T (&)[3], const T (&uo)[3],
                        double (&acc)[2], const Pre& p) const {
        double zi[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const T ax = ((cl >> c) & 1) ? uo[c] : yK[c];
            T dd = c1 * p.di[c] * (p.b[c] - ax);
            if (d) dd = fma(c0, p.d[c], dd);
            zi[c] = (double)(uo[c] + dd);
            acc[0] = fma(zi[c], p.r[c], acc[0]);
            if (!first) acc[1] = fma(zi[c], p.q[c], acc[1]);
        }
        st3(z, b, i, zi);
    }
    __device__ void prologue() {}
    __device__ void done(double (&acc)[2]) const { write_partials<2>(acc, part); }
};

struct EpiSplit {  // yk = N.K(N u), ym = N.M(N u)
    static constexpr int outputs = 2;
    static constexpr bool uses_input = false;
    double* yk;
    double* ym;
    TT_NO_PRE
    __device__ void put(size_t b, const LaneOff& i, uint8_t cl, const double (&yK)[3], const double (&yM)[3],
                        const double (&)[3], double (&)[2], const Pre&) const {
        double k[3], m[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const bool clamped = (cl >> c) & 1;
            k[c] = clamped ? 0.0 : yK[c];
            m[c] = clamped ? 0.0 : yM[c];
        }
        st3(yk, b, i, k);
        st3(ym, b, i, m);
    }
    __device__ void prologue() {}
    __device__ void done(double (&)[2]) const {}
};

struct EpiRaw {  // y = yK + yM, no BC
    static constexpr int outputs = 1;
    static constexpr bool uses_input = false;
    double* y;
    TT_NO_PRE
    __device__ void put(size_t b, const LaneOff& i, uint8_t, const double (&yK)[3], const double (&)[3], const double (&)[3],
                        double (&)[2], const Pre&) const {
        st3(y, b, i, yK);
    }
    __device__ void prologue() {}
    __device__ void done(double (&)[2]) const {}
};

struct EpiRHS {  // R = N.(fs F + yK + yM)
    static constexpr int outputs = 1;
    static constexpr bool uses_input = false;
    const double* F;
    double fs;
    double* R;
    struct Pre {
        double F[3];
    };
    template <class S>
    __device__ __forceinline__ void fetch(size_t b, const LaneOff& i, const S&, Pre& p) const { ld3(F, b, i, p.F); }
    __device__ void put(size_t b, const LaneOff& i, uint8_t cl, const double (&yK)[3], const double (&)[3],
                        const double (&)[3], double (&)[2], const Pre& p) const {
        double v[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            v[c] = ((cl >> c) & 1) ? 0.0 : fma(fs, p.F[c], yK[c]);
        }
        st3(R, b, i, v);
    }
    __device__ void prologue() {}
    __device__ void done(double (&)[2]) const {}
};

// beta of the flexible CG (Polak-Ribiere form) from the z.r and z.q_old partials, formed by every block of a consumer
// (fixed order: bit-identical); block 0 also keeps gamma = z.r for the update.  beta is 0 on a (re)start, and once
// the solve is frozen, when gamma_old may be 0.  (One block for it alone took 4.4 us per iteration; summing ~500
// partials in every block hides behind the other blocks' work.)
__device__ __forceinline__ double fcg_beta(const double* part, int nblk, double* scal, int first) {
    const double done = scal[SC_DONE], al = scal[SC_ALPHA], old = scal[SC_GAMMA_OLD];  // (in flight with the partials)
    double d[2];
    sum_partials<2>(part, nblk, d);
    if (blockIdx.x == 0 && threadIdx.x == 0) scal[SC_GAMMA] = d[0];
    return (first || done != 0.0) ? 0.0 : -al * d[1] / old;
}

// Flexible-CG direction and its product, with z staged (A z from the contraction): p = z + beta p_old,
// q = A p = A z + beta q_old (p_old, q_old read at the owned node), partials of p.q.
struct EpiFcg {
    static constexpr int outputs = 1;
    static constexpr bool uses_input = true;
    double* pnew;
    double* q;
    const double* pold;
    const double* qold;
    double* scal;
    const double* dots;
    int dots_nblk;
    int first;
    double* part;
    double beta;
    struct Pre {
        double p[3], q[3];
    };
    __device__ __forceinline__ void prologue() { beta = fcg_beta(dots, dots_nblk, scal, first); }
    template <class S>
    __device__ __forceinline__ void fetch(size_t b, const LaneOff& i, const S&, Pre& pr) const {
        if (!first) {
            ld3(pold, b, i, pr.p);
            ld3(qold, b, i, pr.q);
        }
    }
    __device__ void put(size_t b, const LaneOff& i, uint8_t cl, const double (&yK)[3], const double (&)[3],
                        const double (&uo)[3], double (&acc)[2], const Pre& pr) const {
        double p[3], v[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const double az = ((cl >> c) & 1) ? uo[c] : yK[c];
            p[c] = first ? uo[c] : fma(beta, pr.p[c], uo[c]);
            v[c] = first ? az : fma(beta, pr.q[c], az);
            acc[0] = fma(p[c], v[c], acc[0]);
        }
        st3(pnew, b, i, p);
        st3(q, b, i, v);
    }
    __device__ void done(double (&acc)[2]) const {
        double a[1] = {acc[0]};
        write_partials<1>(a, part);
    }
};
#undef TT_NO_PRE

template <typename T, typename CT, bool MASKIN, class Stage, class Epi>
static int launch_cols_ct(const OpLevel& L, double cK, double cM, const Stage& st, const Epi& epi, hipStream_t s) {
    const ColSplit& cs = sizeof(T) == 8 ? L.split64 : L.split32;
    const ColPlan& p = cs.plan;
    const ModeConst<T>* mc = sizeof(T) == 8 ? (const ModeConst<T>*)L.modes64 : (const ModeConst<T>*)L.modes32;
    if (p.cx == 0) {  // a small grid
        const int tx = (L.g.nx + 3) / 4, ty = (L.g.ny + 3) / 4, tz = (L.g.nz + 3) / 4;
        hipLaunchKernelGGL((k_apply_box<T, CT, MASKIN, Stage, Epi>), dim3(tx * ty * tz), dim3(128), 0, s, gargs(L.g), tx,
                           ty, mc, (const CT*)L.kf, (const CT*)L.mf, (T)cK, (T)cM, L.mask, st, epi);
        TT_HIP(hipGetLastError());
        return tx * ty * tz;
    }
    const int nb = 8 * ((p.ntiles() + 7) / 8);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(nb), dim3(256), 0, s, gargs(L.g), (const ColTile&)p, mc, (const CT*)L.kf,
                           (const CT*)L.mf, (T)cK, (T)cM, L.mask, cs.bc, st, epi, p.strands);
    };
    if (p.strands > 1) launch(k_apply_cols<T, CT, MASKIN, true, Stage, Epi>);
    else launch(k_apply_cols<T, CT, MASKIN, false, Stage, Epi>);
    TT_HIP(hipGetLastError());
    return nb;
}
// launch on the level's coefficient kind; returns the block count (= number of reduction partials)
template <typename T, bool MASKIN, class Stage, class Epi>
static int run_apply(const OpLevel& L, double cK, double cM, const Stage& st, const Epi& epi, hipStream_t s) {
    switch (L.coef_kind) {
    case COEF_F64: return launch_cols_ct<T, double, MASKIN>(L, cK, cM, st, epi, s);
    case COEF_F32: return launch_cols_ct<T, float, MASKIN>(L, cK, cM, st, epi, s);
    default: return launch_cols_ct<T, bf16_t, MASKIN>(L, cK, cM, st, epi, s);
    }
}

// the blocks of an apply launch on this level must fit the reducer's partial regions
static inline void check_partials(const OpLevel& L, const Reducer& red) {
    const int nt = std::max(L.split64.plan.blocks(), L.split32.plan.blocks());
    TT_CHECK(nt <= red.maxblocks, -3, "reducer too small");
}

void launch_apply_bc(const OpLevel& L, double cK, double cM, const void* u, void* y, bool fp64, hipStream_t s,
                     Reducer* red, int dot_slot) {
    if (fp64) {
        StageOne<double> st{(const double*)u};
        if (red) {
            check_partials(L, *red);
            EpiBCDot<double> e{(double*)y, red->part(dot_slot)};
            red->nblk[dot_slot] = run_apply<double, true>(L, cK, cM, st, e, s);
            red->nv[dot_slot] = 1;
        } else {
            run_apply<double, true>(L, cK, cM, st, EpiBC<double>{(double*)y}, s);
        }
    } else {
        StageOne<float> st{(const float*)u};
        if (red) {
            check_partials(L, *red);
            EpiBCDot<float> e{(float*)y, red->part(dot_slot)};
            red->nblk[dot_slot] = run_apply<float, true>(L, cK, cM, st, e, s);
            red->nv[dot_slot] = 1;
        } else {
            run_apply<float, true>(L, cK, cM, st, EpiBC<float>{(float*)y}, s);
        }
    }
}

void launch_residual(const OpLevel& L, double cK, double cM, const void* b, const void* x, void* r, bool fp64,
                     hipStream_t s) {
    if (fp64)
        run_apply<double, true>(L, cK, cM, StageOne<double>{(const double*)x},
                                       EpiResid<double>{(const double*)b, (double*)r}, s);
    else
        run_apply<float, true>(L, cK, cM, StageOne<float>{(const float*)x},
                                      EpiResid<float>{(const float*)b, (float*)r}, s);
}

void launch_resid_first(const OpLevel& L, double cK, double cM, const void* b, const void* dinv, double c1, void* x,
                        void* r, bool fp64, hipStream_t s) {
    if (fp64)
        run_apply<double, true>(
            L, cK, cM, StageChebFirst<double, false>{nullptr, (const double*)b, (const double*)dinv, c1},
            EpiResidFirst<double>{(double*)x, (double*)r}, s);
    else
        run_apply<float, true>(
            L, cK, cM, StageChebFirst<float, false>{nullptr, (const float*)b, (const float*)dinv, (float)c1},
            EpiResidFirst<float>{(float*)x, (float*)r}, s);
}

void launch_residual_dots(const OpLevel& L, double cK, double cM, const double* b, const double* x, double* r,
                          Reducer& red, int bb_region, int rr_region, hipStream_t s) {
    check_partials(L, red);
    EpiResidDots e{b, r, red.part(bb_region), red.part(rr_region)};
    const int nb = run_apply<double, true>(L, cK, cM, StageOne<double>{x}, e, s);
    red.nblk[bb_region] = red.nblk[rr_region] = nb;
    red.nv[bb_region] = red.nv[rr_region] = 1;
}

void launch_cheb_step(const OpLevel& L, double cK, double cM, const void* b, const void* x, const void* d,
                      const void* dinv, double c0, double c1, void* xn, void* dn, bool fp64, hipStream_t s) {
    if (fp64) {
        EpiCheb<double> e{(const double*)b, (const double*)d, (const double*)dinv, c0, c1, (double*)xn, (double*)dn};
        run_apply<double, true>(L, cK, cM, StageOne<double>{(const double*)x}, e, s);
    } else {
        EpiCheb<float> e{(const float*)b,  (const float*)d, (const float*)dinv, (float)c0,
                         (float)c1,        (float*)xn,      (float*)dn};
        run_apply<float, true>(L, cK, cM, StageOne<float>{(const float*)x}, e, s);
    }
}

void launch_cheb_first_step(const OpLevel& L, double cK, double cM, const double* r64, void* b, const void* dinv,
                            double c1_first, double c0, double c1, void* xn, void* dn, bool fp64, hipStream_t s) {
    if (fp64) {
        const double* dv = (const double*)dinv;
        if (r64)
            run_apply<double, true>(L, cK, cM, StageChebFirst<double, true>{r64, nullptr, dv, c1_first},
                                           EpiChebFirst<double, true>{(double*)b, dv, c0, c1, (double*)xn,
                                                                      (double*)dn}, s);
        else
            run_apply<double, true>(L, cK, cM,
                                           StageChebFirst<double, false>{nullptr, (const double*)b, dv, c1_first},
                                           EpiChebFirst<double, false>{nullptr, dv, c0, c1, (double*)xn,
                                                                       (double*)dn}, s);
    } else {
        const float* dv = (const float*)dinv;
        if (r64)
            run_apply<float, true>(L, cK, cM, StageChebFirst<float, true>{r64, nullptr, dv, (float)c1_first},
                                          EpiChebFirst<float, true>{(float*)b, dv, (float)c0, (float)c1,
                                                                    (float*)xn, (float*)dn}, s);
        else
            run_apply<float, true>(L, cK, cM,
                                          StageChebFirst<float, false>{nullptr, (const float*)b, dv, (float)c1_first},
                                          EpiChebFirst<float, false>{nullptr, dv, (float)c0, (float)c1, (float*)xn,
                                                                     (float*)dn}, s);
    }
}

void launch_cheb_last(const OpLevel& L, double cK, double cM, const void* b, const void* x, const void* d,
                      const void* dinv, double c0, double c1, double* z, const double* r, const double* q, bool first,
                      bool fp64, Reducer& red, hipStream_t s) {
    check_partials(L, red);
    if (fp64) {
        EpiChebOut<double> e{(const double*)b, (const double*)d, (const double*)dinv, c0, c1, z, r, q,
                             first ? 1 : 0, red.part(PB_DOTS)};
        red.nblk[PB_DOTS] = run_apply<double, true>(L, cK, cM, StageOne<double>{(const double*)x}, e, s);
    } else {
        EpiChebOut<float> e{(const float*)b, (const float*)d, (const float*)dinv, (float)c0, (float)c1, z, r, q,
                            first ? 1 : 0, red.part(PB_DOTS)};
        red.nblk[PB_DOTS] = run_apply<float, true>(L, cK, cM, StageOne<float>{(const float*)x}, e, s);
    }
    red.nv[PB_DOTS] = 2;
}

void launch_apply_split(const OpLevel& L, double cK, double cM, const double* u, double* yk, double* ym,
                        hipStream_t s) {
    run_apply<double, true>(L, cK, cM, StageOne<double>{u}, EpiSplit{yk, ym}, s);
}

void launch_apply_raw(const OpLevel& L, const double* kf, const double* mf, double cK, double cM, const double* u,
                      double* y, hipStream_t s) {
    OpLevel L2 = L;
    L2.kf = kf;
    L2.mf = mf;
    L2.coef_kind = COEF_F64;
    run_apply<double, false>(L2, cK, cM, StageOne<double>{u}, EpiRaw{y}, s);
}

void launch_newmark_rhs(const OpLevel& L, const double* u, const double* v, const double* a, const double* F,
                        double fs, const double wK[3], const double wM[3], double* R, hipStream_t s) {
    StageThree st{u, v, a, wK[0], wK[1], wK[2], wM[0], wM[1], wM[2]};
    run_apply<double, true>(L, 1.0, 1.0, st, EpiRHS{F, fs, R}, s);
}

// single-block reductions of partials: 1024 threads, so each sums ~5 of the ~5000 partials of a
// fine-grid launch (latency bound: 256 threads took ~4.6 us per call)
constexpr int BSR = 1024;
void launch_fcg_apply(const OpLevel& L, double cK, double cM, const double* z, const double* p_old, double* p_new,
                      const double* q_old, double* q_new, Reducer& red, bool first, hipStream_t s) {
    check_partials(L, red);
    EpiFcg e{p_new, q_new,        p_old, q_old, red.scal.p, red.part(PB_DOTS), red.nblk[PB_DOTS], first ? 1 : 0,
             red.part(PB_PQ), 0.0};
    red.nblk[PB_PQ] = run_apply<double, true>(L, cK, cM, StageOne<double>{z}, e, s);
    red.nv[PB_PQ] = 1;
}

// ------------------------------------------------------------------ diagonal
template <typename T, typename CT>
__global__ void k_diag_inv(GridArgs g, const double* __restrict__ KE, const double* __restrict__ M8,
                           const CT* __restrict__ kf, const CT* __restrict__ mf, double cK, double cM,
                           const uint8_t* __restrict__ mask, T* __restrict__ dinv) {
    const long n = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (n >= (long)g.nx * g.ny * g.nz) return;
    const int i = n % g.nx, j = (n / g.nx) % g.ny, k = n / ((long)g.nx * g.ny);
    double d[3] = {0, 0, 0};
    for (int ez = 0; ez < 2; ez++)
        for (int ey = 0; ey < 2; ey++)
            for (int ex = 0; ex < 2; ex++) {
                const int ei = i - 1 + ex, ej = j - 1 + ey, ek = k - 1 + ez;
                if (ei < 0 || ej < 0 || ek < 0 || ei >= g.ex || ej >= g.ey || ek >= g.ez) continue;
                const long e = ei + (long)g.ex * (ej + (long)g.ey * ek);
                const int a = corner_id(1 - ex, 1 - ey, 1 - ez);
                const double kk = cK * coef_ld(kf, e), mm = cM * coef_ld(mf, e);
                for (int c = 0; c < 3; c++) d[c] += kk * KE[(3 * a + c) * 25] + mm * M8[a * 9];
            }
    const uint8_t cl = mask[n];
    for (int c = 0; c < 3; c++) dinv[3 * n + c] = (T)(((cl >> c) & 1) ? 1.0 : 1.0 / d[c]);
}

void launch_diag_inv(const OpLevel& L, double cK, double cM, void* dinv, bool fp64, hipStream_t s) {
    GridArgs ga = gargs(L.g);
    int nb = nblocks(L.g.nn);
#define TT_DIAG(T, CT) \
    hipLaunchKernelGGL((k_diag_inv<T, CT>), dim3(nb), dim3(BS), 0, s, ga, L.KE64, L.M864, (const CT*)L.kf, (const CT*)L.mf, cK, cM, L.mask, (T*)dinv)
    if (fp64) {
        if (L.coef_kind == COEF_F64) TT_DIAG(double, double);
        else if (L.coef_kind == COEF_F32) TT_DIAG(double, float);
        else TT_DIAG(double, bf16_t);
    } else {
        if (L.coef_kind == COEF_F64) TT_DIAG(float, double);
        else if (L.coef_kind == COEF_F32) TT_DIAG(float, float);
        else TT_DIAG(float, bf16_t);
    }
#undef TT_DIAG
    TT_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ vector kernels
template <typename T>
__global__ void k_fill(T* x, T v, long n) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) x[i] = v;
}
void launch_fill(void* x, double v, long n, bool fp64, hipStream_t s) {
    if (n <= 0) return;
    if (fp64) hipLaunchKernelGGL(k_fill<double>, dim3(nblocks(n)), dim3(BS), 0, s, (double*)x, v, n);
    else hipLaunchKernelGGL(k_fill<float>, dim3(nblocks(n)), dim3(BS), 0, s, (float*)x, (float)v, n);
    TT_HIP(hipGetLastError());
}

// x_i uniform in [-1, 1) from a counter-based hash of (seed, i) (splitmix64 finaliser): a deterministic
// start vector made on the device, with no host loop or copy
template <typename T>
__global__ void k_fill_hash(T* __restrict__ x, long n, unsigned long long seed) {
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    unsigned long long z = seed + 0x9E3779B97F4A7C15ull * (unsigned long long)(i + 1);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    x[i] = (T)((double)(z >> 11) * (2.0 / 9007199254740992.0) - 1.0);
}
void launch_fill_hash(void* x, long n, unsigned long long seed, bool fp64, hipStream_t s) {
    if (n <= 0) return;
    if (fp64) hipLaunchKernelGGL(k_fill_hash<double>, dim3(nblocks(n)), dim3(BS), 0, s, (double*)x, n, seed);
    else hipLaunchKernelGGL(k_fill_hash<float>, dim3(nblocks(n)), dim3(BS), 0, s, (float*)x, n, seed);
    TT_HIP(hipGetLastError());
}

// x = N.x: dof c of node n is zeroed where bit c of mask[n] is set
__global__ void k_mask_dofs(double* __restrict__ x, const uint8_t* __restrict__ mask, long nd) {
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < nd && ((mask[i / 3] >> (i % 3)) & 1)) x[i] = 0.0;
}
void launch_mask_dofs(double* x, const uint8_t* mask, long nd, hipStream_t s) {
    if (nd <= 0) return;
    hipLaunchKernelGGL(k_mask_dofs, dim3(nblocks(nd)), dim3(BS), 0, s, x, mask, nd);
    TT_HIP(hipGetLastError());
}

template <typename S, typename D>
__global__ void k_copy(const S* __restrict__ a, D* __restrict__ b, long n) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) b[i] = (D)a[i];
}
void launch_copy(const void* src, void* dst, long n, bool s64, bool d64, hipStream_t s) {
    if (n <= 0) return;
    dim3 gr(nblocks(n)), bl(BS);
    if (s64 && d64) hipLaunchKernelGGL((k_copy<double, double>), gr, bl, 0, s, (const double*)src, (double*)dst, n);
    else if (s64) hipLaunchKernelGGL((k_copy<double, float>), gr, bl, 0, s, (const double*)src, (float*)dst, n);
    else if (d64) hipLaunchKernelGGL((k_copy<float, double>), gr, bl, 0, s, (const float*)src, (double*)dst, n);
    else hipLaunchKernelGGL((k_copy<float, float>), gr, bl, 0, s, (const float*)src, (float*)dst, n);
    TT_HIP(hipGetLastError());
}

template <typename T>
__global__ void k_cheb_first(const T* __restrict__ b, const T* __restrict__ dinv, T c1, T* __restrict__ x, long n) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) x[i] = c1 * dinv[i] * b[i];
}
// b = (T) r (FP64 in) and x = c1 D^-1 b: the start of a V-cycle on the finest level
template <typename T>
__global__ void k_cheb_first_from64(const double* __restrict__ r, T* __restrict__ b, const T* __restrict__ dinv, T c1,
                                    T* __restrict__ x, long n) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) {
        const T bi = (T)r[i];
        b[i] = bi;
        x[i] = c1 * dinv[i] * bi;
    }
}
void launch_cheb_first_from64(const double* r, void* b, const void* dinv, double c1, void* x, long n, bool fp64,
                              hipStream_t s) {
    if (fp64)
        hipLaunchKernelGGL(k_cheb_first_from64<double>, dim3(nblocks(n)), dim3(BS), 0, s, r, (double*)b,
                           (const double*)dinv, c1, (double*)x, n);
    else
        hipLaunchKernelGGL(k_cheb_first_from64<float>, dim3(nblocks(n)), dim3(BS), 0, s, r, (float*)b,
                           (const float*)dinv, (float)c1, (float*)x, n);
    TT_HIP(hipGetLastError());
}

void launch_cheb_first(const void* b, const void* dinv, double c1, void* x, long n, bool fp64, hipStream_t s) {
    if (fp64)
        hipLaunchKernelGGL(k_cheb_first<double>, dim3(nblocks(n)), dim3(BS), 0, s, (const double*)b,
                           (const double*)dinv, c1, (double*)x, n);
    else
        hipLaunchKernelGGL(k_cheb_first<float>, dim3(nblocks(n)), dim3(BS), 0, s, (const float*)b,
                           (const float*)dinv, (float)c1, (float*)x, n);
    TT_HIP(hipGetLastError());
}

// restriction R = P^T of trilinear interpolation (PETSc DMDA Q1 interpolation, LinearElasticity.cc:2840-2844).
// Branch-free and fully unrolled so that the 27 neighbour loads are in flight together: neighbours
// outside the fine grid get weight 0 at a clamped (valid) index, which leaves the sum unchanged.
// The coarse output may be wider than the fine input (FP32 levels feeding an FP64 coarsest solve).
// NC: components per thread.  A node per thread (3) where the coarse grid has enough nodes to fill the chip: one wide load
// per neighbour; a dof per thread (1) below, where more and shorter chains of loads are what counts: at 225 coarse nodes
// 2.8 instead of 4.6 us (FP64), at 35,937 4.7 instead of 3.9 us (FP32).  Blocks of one wave (3): the grid is about one wave
// per SIMD, and 277 blocks of 256 left a second round on 21 CUs (70,785 coarse nodes: FP32 8.7 -> 6.1 us, FP64 9.0 -> 7.1).
template <int NC, typename Tf, typename Tc>
__global__ void k_restrict(GridArgs f, GridArgs c, const Tf* __restrict__ rf, const uint8_t* __restrict__ cmask,
                           Tc* __restrict__ bc) {
    const unsigned t = blockIdx.x * blockDim.x + threadIdx.x, n = NC == 3 ? t : t / 3u, q = NC == 3 ? 0u : t - 3u * n;
    if (n >= (unsigned)(c.nx * c.ny * c.nz)) return;
    int I, J, K;
    grid_ijk(n, c.nx, c.ny, I, J, K);
    const uint8_t cl = cmask[n];
    Tf s[NC];
#pragma unroll
    for (int d = 0; d < NC; d++) s[d] = 0;
#pragma unroll
    for (int dk = -1; dk <= 1; dk++) {
        const int k = 2 * K + dk;
        const bool kin = k >= 0 && k < f.nz;
        const Tf wk = kin ? (dk == 0 ? (Tf)1 : (Tf)0.5) : (Tf)0;
        const int kc = kin ? k : 2 * K;
#pragma unroll
        for (int dj = -1; dj <= 1; dj++) {
            const int j = 2 * J + dj;
            const bool jin = j >= 0 && j < f.ny;
            const Tf wj = jin ? (dj == 0 ? wk : wk * (Tf)0.5) : (Tf)0;
            const int jc = jin ? j : 2 * J;
#pragma unroll
            for (int di = -1; di <= 1; di++) {
                const int i = 2 * I + di;
                const bool iin = i >= 0 && i < f.nx;
                const Tf w = iin ? (di == 0 ? wj : wj * (Tf)0.5) : (Tf)0;
                const int ic = iin ? i : 2 * I;
                const unsigned m = (unsigned)ic + (unsigned)f.nx * ((unsigned)jc + (unsigned)f.ny * (unsigned)kc);
#pragma unroll
                for (int d = 0; d < NC; d++) s[d] = fma(w, rf[3u * m + q + d], s[d]);
            }
        }
    }
#pragma unroll
    for (int d = 0; d < NC; d++) bc[3u * n + q + d] = ((cl >> (q + d)) & 1) ? (Tc)0 : (Tc)s[d];
}
void launch_restrict(const Grid& fine, const Grid& coarse, const void* rf, const uint8_t* cmask, void* bc, bool fp64,
                     bool out64, hipStream_t s) {
    auto launch = [&](auto kernel, int nc, auto* src, auto* dst) {
        const int bs = nc == 3 ? 64 : 128;
        hipLaunchKernelGGL(kernel, dim3(nblocks(3 / nc * coarse.nn, bs)), dim3(bs), 0, s, gargs(fine), gargs(coarse), src,
                           cmask, dst);
    };
    const bool small = coarse.nn <= 16384;
    if (fp64) {
        if (small) launch(k_restrict<1, double, double>, 1, (const double*)rf, (double*)bc);
        else launch(k_restrict<3, double, double>, 3, (const double*)rf, (double*)bc);
    } else if (out64) {
        if (small) launch(k_restrict<1, float, double>, 1, (const float*)rf, (double*)bc);
        else launch(k_restrict<3, float, double>, 3, (const float*)rf, (double*)bc);
    } else {
        if (small) launch(k_restrict<1, float, float>, 1, (const float*)rf, (float*)bc);
        else launch(k_restrict<3, float, float>, 3, (const float*)rf, (float*)bc);
    }
    TT_HIP(hipGetLastError());
}

// xf += P_1 x_1 + P_2 x_2 + ... on free dofs: the corrections of one or several coarser levels, each interpolated to the
// fine nodes directly.  Nested trilinear interpolation is trilinear on the coarser cells, and a level's clamped dofs lie
// on faces and edges whose coarse nodes are clamped (zero) too, so a chain of prolongations through the levels between,
// x_1 += P x_2 and then xf += P x_1, is this sum: one kernel per V-cycle instead of one per level where the
// intermediate levels do not smooth after the correction.  Level l's node of fine node i is i >> l with weight
// (1 - f), f = (i mod 2^l) / 2^l, and its successor with f (at a valid index when f = 0).  At 128x64x64 (4 levels) 7.0 +
// 4.0 + 3.4 us for the three kernels before.
struct ProlongChain {
    const void* x[7];
    int nx[7], ny[7], nz[7];
    int n;
};
// adds level l's correction at the fine nodes (i, j + b, k + d), b < 2, d < NZ (s[b + 2 d]), j (and k with NZ = 2) even: all
// lie in one cell of every coarser level
template <int NZ, typename Tf, typename Tx>
__device__ __forceinline__ void prolong_level(const Tx* __restrict__ x, int nx, int ny, int nz, int l, int i, int j, int k,
                                              Tf (&s)[2 * NZ][3]) {
    const Tf inv = (Tf)1 / (Tf)(1 << l);
    const int fi = i & ((1 << l) - 1), fj = j & ((1 << l) - 1), fk = k & ((1 << l) - 1);
    const Tf wi = (Tf)fi * inv;
    const int di = fi ? 3 : 0, dj = (j >> l) + 1 < ny ? 3 * nx : 0;
    const int dk = (NZ == 2 ? (k >> l) + 1 < nz : fk != 0) ? 3 * nx * ny : 0;
    const Tx* p = x + 3 * ((size_t)(i >> l) + (size_t)nx * ((j >> l) + (size_t)ny * (k >> l)));
    Tf v[2][2][3];  // the cell's edges in x at i: [z][y]
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const Tx* pq = p + ((q & 1) ? dj : 0) + ((q & 2) ? dk : 0);
#pragma unroll
        for (int c = 0; c < 3; c++) v[q >> 1][q & 1][c] = fma((Tf)1 - wi, (Tf)pq[c], wi * (Tf)pq[di + c]);
    }
#pragma unroll
    for (int b = 0; b < 2; b++) {
        const Tf wj = (Tf)(fj + b) * inv;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const Tf lo = fma((Tf)1 - wj, v[0][0][c], wj * v[0][1][c]), hi = fma((Tf)1 - wj, v[1][0][c], wj * v[1][1][c]);
#pragma unroll
            for (int d = 0; d < NZ; d++) {
                const Tf wk = (Tf)(fk + d) * inv;
                s[b + 2 * d][c] = fma((Tf)1 - wk, lo, fma(wk, hi, s[b + 2 * d][c]));
            }
        }
    }
}
// Tl: the last (coarsest) level's type; one thread per two nodes in y (and NZ in z), the lanes of a wave along x, so that
// the fine vector is read and written in order and neighbouring lanes share the coarse loads: the kernel is bound by
// its memory instructions.  128x64x64, 3 coarser levels: 11.8 us (FP32) and 16.4 us (FP64) with two nodes in x per
// thread, 10.4 and 15.0 with NZ = 1, 8.5 and 13.4 with NZ = 2.  NZ = 2 takes grids above kChainNodes: at 70,785 nodes
// (64x32x32) NZ = 1 and 2 take 5.6 and 5.6 us (FP32), 6.1 and 7.2 (FP64), at 1,377 (16x8x8) 3.6 and 4.0, at 232,897
// (96x48x48, FP32) 6.5 and 5.9.  Blocks of one wave even out the CUs (9.1 -> 8.7 us on one box, 3.4 -> 3.1 at 16x8x8).
constexpr long kChainNodes = 131072;
template <int NZ, typename Tf, typename Tl>
__global__ void k_prolong_chain(GridArgs f, ProlongChain pc, const uint8_t* __restrict__ fmask, Tf* __restrict__ xf) {
    const unsigned py = (unsigned)(f.ny + 1) >> 1, pz = (unsigned)(f.nz + NZ - 1) / NZ;
    const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (t >= (long)f.nx * py * pz) return;
    int i, j, k;
    grid_ijk((unsigned)t, f.nx, py, i, j, k);
    j *= 2;
    k *= NZ;
    // (a node beyond the grid is read as the one before it and not written)
    const long oy = j + 1 < f.ny ? f.nx : 0, oz = NZ == 2 && k + 1 < f.nz ? (long)f.nx * f.ny : 0;
    const long n = i + (long)f.nx * (j + (long)f.ny * k);
    uint8_t cl[2 * NZ];
    Tf x[2 * NZ][3], s[2 * NZ][3] = {};
#pragma unroll
    for (int q = 0; q < 2 * NZ; q++) {
        const long m = n + ((q & 1) ? oy : 0) + ((q & 2) ? oz : 0);
        cl[q] = ((q & 1) && !oy) || ((q & 2) && !oz) ? (uint8_t)7 : fmask[m];
#pragma unroll
        for (int c = 0; c < 3; c++) x[q][c] = xf[3 * m + c];
    }
    for (int l = 0; l + 1 < pc.n; l++)
        prolong_level<NZ, Tf, Tf>((const Tf*)pc.x[l], pc.nx[l], pc.ny[l], pc.nz[l], l + 1, i, j, k, s);
    const int l = pc.n - 1;
    prolong_level<NZ, Tf, Tl>((const Tl*)pc.x[l], pc.nx[l], pc.ny[l], pc.nz[l], l + 1, i, j, k, s);
#pragma unroll
    for (int q = 0; q < 2 * NZ; q++) {
        const long m = n + ((q & 1) ? oy : 0) + ((q & 2) ? oz : 0);
#pragma unroll
        for (int c = 0; c < 3; c++)
            if (!((cl[q] >> c) & 1)) xf[3 * m + c] = x[q][c] + s[q][c];
    }
}
void launch_prolong_chain(const Grid& fine, int n, const Grid* const* coarse, const void* const* xc,
                          const uint8_t* fmask, void* xf, bool fp64, bool last64, hipStream_t s) {
    TT_CHECK(n >= 1 && n <= 7, -3, "launch_prolong_chain: 1..7 levels");
    ProlongChain pc{};
    pc.n = n;
    for (int l = 0; l < n; l++) {
        pc.x[l] = xc[l];
        pc.nx[l] = coarse[l]->nx;
        pc.ny[l] = coarse[l]->ny;
        pc.nz[l] = coarse[l]->nz;
    }
    auto launch = [&](auto kernel, int nz, auto* x) {
        const long threads = (long)fine.nx * ((fine.ny + 1) / 2) * ((fine.nz + nz - 1) / nz);
        hipLaunchKernelGGL(kernel, dim3(nblocks(threads, 64)), dim3(64), 0, s, gargs(fine), pc, fmask, x);
    };
    const bool big = fine.nn > kChainNodes;
    if (fp64) {
        if (big) launch(k_prolong_chain<2, double, double>, 2, (double*)xf);
        else launch(k_prolong_chain<1, double, double>, 1, (double*)xf);
    } else if (last64) {
        if (big) launch(k_prolong_chain<2, float, double>, 2, (float*)xf);
        else launch(k_prolong_chain<1, float, double>, 1, (float*)xf);
    } else {
        if (big) launch(k_prolong_chain<2, float, float>, 2, (float*)xf);
        else launch(k_prolong_chain<1, float, float>, 1, (float*)xf);
    }
    TT_HIP(hipGetLastError());
}

// rediscretised coarse coefficients: mean of the 8 child elements
__global__ void k_coarsen_coef(GridArgs f, GridArgs c, const double* __restrict__ kff, const double* __restrict__ mff,
                               double* __restrict__ kfc, double* __restrict__ mfc) {
    const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (e >= (long)c.ex * c.ey * c.ez) return;
    const int I = e % c.ex, J = (e / c.ex) % c.ey, K = e / ((long)c.ex * c.ey);
    double sk = 0.0, sm = 0.0;
    for (int dk = 0; dk < 2; dk++)
        for (int dj = 0; dj < 2; dj++)
            for (int di = 0; di < 2; di++) {
                const long fe = (2 * I + di) + (long)f.ex * ((2 * J + dj) + (long)f.ey * (2 * K + dk));
                sk += kff[fe];
                sm += mff[fe];
            }
    kfc[e] = 0.125 * sk;
    mfc[e] = 0.125 * sm;
}
void launch_coarsen_coef(const Grid& fine, const Grid& coarse, const double* kf_f, const double* mf_f, double* kf_c,
                         double* mf_c, hipStream_t s) {
    hipLaunchKernelGGL(k_coarsen_coef, dim3(nblocks(coarse.nel)), dim3(BS), 0, s, gargs(fine), gargs(coarse), kf_f,
                       mf_f, kf_c, mf_c);
    TT_HIP(hipGetLastError());
}

__device__ __forceinline__ bf16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
    return (bf16_t)(u >> 16);
}
__global__ void k_convert_coef(const double* __restrict__ src, void* dst, long n, int kind) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (kind == COEF_F32) ((float*)dst)[i] = (float)src[i];
    else if (kind == COEF_BF16) ((bf16_t*)dst)[i] = f2bf((float)src[i]);
    else ((double*)dst)[i] = src[i];
}
void launch_convert_coef(const double* src, void* dst, long n, int kind, hipStream_t s) {
    hipLaunchKernelGGL(k_convert_coef, dim3(nblocks(n)), dim3(BS), 0, s, src, dst, n, kind);
    TT_HIP(hipGetLastError());
}

// SIMP / RAMP / linear interpolation (LinearElasticity.cc:1580-1623)
__device__ __forceinline__ void interp1(int scheme, double vmin, double vmax, double p, double x, double& f,
                                        double& df) {
    if (scheme == 0) {
        f = vmin + x * (vmax - vmin);
        df = vmax - vmin;
    } else if (scheme == 1) {
        f = vmin + pow(x, p) * (vmax - vmin);
        df = p * pow(x, p - 1) * (vmax - vmin);
    } else {
        f = vmin + x / (1 + p * (1 - x)) * (vmax - vmin);
        df = (1 + p) / pow(1 + p * (1 - x), 2) * (vmax - vmin);
    }
}
__global__ void k_interp(const double* __restrict__ x, long n, int sInt, double Emin, double Emax, double pK, int mInt,
                         double Rmin, double Rmax, double pM, const double* __restrict__ P, double* kf, double* mf,
                         double* dkf, double* dmf, double* Pkf, double* Pmf) {
    long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (e >= n) return;
    double k, dk, m, dm;
    interp1(sInt, Emin, Emax, pK, x[e], k, dk);
    interp1(mInt, Rmin, Rmax, pM, x[e], m, dm);
    kf[e] = k;
    mf[e] = m;
    dkf[e] = dk;
    dmf[e] = dm;
    Pkf[e] = P[e] * k;
    Pmf[e] = P[e] * m;
}
void launch_interp(const double* x, long n, int sInt, double Emin, double Emax, double pK, int mInt, double Rmin,
                   double Rmax, double pM, const double* P, double* kf, double* mf, double* dkf, double* dmf,
                   double* Pkf, double* Pmf, hipStream_t s) {
    hipLaunchKernelGGL(k_interp, dim3(nblocks(n)), dim3(BS), 0, s, x, n, sInt, Emin, Emax, pK, mInt, Rmin, Rmax, pM,
                       P, kf, mf, dkf, dmf, Pkf, Pmf);
    TT_HIP(hipGetLastError());
}

// In-place inverse of an m x m (m <= 64) symmetric positive definite block (column-major, leading
// dimension lda) by the symmetric sweep: step k, with p = 1 / a_kk, sets a_ij -= a_ik a_jk p (i, j != k),
// a_ik *= p (i != k) and a_kk = -p; the matrix stays symmetric, and after all m steps it holds -A^-1.
// 256 threads: thread t holds rows 16 (t / 64) .. + 15 of column t % 64 in registers; the owner lanes
// put column k in LDS for each step (double-buffered, one barrier per step).  A pivot that is not
// positive sets *info.
__global__ __launch_bounds__(256) void k_spd_inv_small(double* A, int m, int lda, int* info) {
    __shared__ double colk[2][64];
    const int t = threadIdx.x, j = t & 63;
    const int rb = __builtin_amdgcn_readfirstlane(t >> 6);  // (wave-uniform: the pivot row's wave branches)
    double c[16];
#pragma unroll
    for (int ii = 0; ii < 16; ii++) {
        const int i = 16 * rb + ii;
        c[ii] = (i < m && j < m) ? A[i + (size_t)j * lda] : 0.0;
    }
    bool bad = false;
    for (int kb = 0; kb < 4; kb++) {
#pragma unroll
        for (int kk = 0; kk < 16; kk++) {
            const int k = 16 * kb + kk;
            if (k < m) {
                double* ck = colk[k & 1];
                if (j == k)
#pragma unroll
                    for (int ii = 0; ii < 16; ii++) ck[16 * rb + ii] = c[ii];
                __syncthreads();
                const double akk = ck[k];
                bad = bad || !(akk > 0.0);
                const double p = 1.0 / akk;
                const double ajk = ck[j] * p;  // a_jk / a_kk (= a_kj / a_kk)
                // c_i -= a_ik a_jk / a_kk; column k itself becomes a_ik p; then the pivot row's element
#pragma unroll
                for (int ii = 0; ii < 16; ii++) c[ii] = fma(-ck[16 * rb + ii], ajk, c[ii]);
                if (j == k)
#pragma unroll
                    for (int ii = 0; ii < 16; ii++) c[ii] = ck[16 * rb + ii] * p;
                if (rb == kb) c[kk] = j == k ? -p : ajk;
            }
        }
    }
    if (bad && t == 0) *info = 1;
#pragma unroll
    for (int ii = 0; ii < 16; ii++) {
        const int i = 16 * rb + ii;
        if (i < m && j < m) A[i + (size_t)j * lda] = -c[ii];
    }
}
void launch_spd_inv_small(double* A, int m, int lda, int* info, hipStream_t s) {
    TT_CHECK(m >= 1 && m <= 64, -3, "launch_spd_inv_small: block of 1..64");  // TT_ERR_INTERNAL
    hipLaunchKernelGGL(k_spd_inv_small, dim3(1), dim3(256), 0, s, A, m, lda, info);
    TT_HIP(hipGetLastError());
}

// dst (cols x rows) = src (rows x cols)^T, both column-major with their leading dimensions
__global__ void k_transpose(const double* __restrict__ src, int rows, int cols, int lds, double* __restrict__ dst,
                            int ldd) {
    __shared__ double t[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8 threads
    const int i0 = blockIdx.x * 32, j0 = blockIdx.y * 32;   // src tile: rows i0.., cols j0..
    for (int r = ty; r < 32; r += 8) {
        const int i = i0 + tx, j = j0 + r;
        if (i < rows && j < cols) t[r][tx] = src[i + (size_t)j * lds];
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        const int i = i0 + r, j = j0 + tx;  // dst (row j, col i) = src (row i, col j)
        if (i < rows && j < cols) dst[j + (size_t)i * ldd] = t[tx][r];
    }
}
void launch_transpose(const double* src, int rows, int cols, int lds, double* dst, int ldd, hipStream_t s) {
    hipLaunchKernelGGL(k_transpose, dim3((rows + 31) / 32, (cols + 31) / 32), dim3(256), 0, s, src, rows, cols, lds,
                       dst, ldd);
    TT_HIP(hipGetLastError());
}
// ---- dense coarsest operator, assembled on the device: entry (i, j) of N (cK K + cM M) N + I - N, i = 3 p + c,
// j = 3 q + d, for the 27 neighbours q of node p (all other entries stay 0 from the clear before).  One
// thread per (i, neighbour, d) sums the element contributions in increasing element order, so the result
// does not depend on scheduling (deterministic set-up).
__global__ void k_dense_coarse(GridArgs g, const double* __restrict__ kf, const double* __restrict__ mf, double cK,
                               double cM, const double* __restrict__ KE, const double* __restrict__ M8,
                               const uint8_t* __restrict__ mask, int n, double* __restrict__ A) {
    const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (t >= (long)n * 81) return;
    const int i = (int)(t / 81), r = (int)(t % 81);
    const int nb = r / 3, d = r % 3;
    const int p = i / 3, c = i % 3;
    const int pi = p % g.nx, pj = (p / g.nx) % g.ny, pk = p / (g.nx * g.ny);
    const int qi = pi + nb % 3 - 1, qj = pj + (nb / 3) % 3 - 1, qk = pk + nb / 9 - 1;
    if (qi < 0 || qi >= g.nx || qj < 0 || qj >= g.ny || qk < 0 || qk >= g.nz) return;
    const int q = qi + g.nx * (qj + g.ny * qk), j = 3 * q + d;
    double val = 0.0;
    if (((mask[p] >> c) & 1) || ((mask[q] >> d) & 1)) {
        val = i == j ? 1.0 : 0.0;
    } else {
        // elements holding both nodes: origin (ei, ej, ek) with max(p, q) - 1 <= e <= min(p, q) per axis
        for (int ek = max(max(pk, qk) - 1, 0); ek <= min(min(pk, qk), g.ez - 1); ek++)
            for (int ej = max(max(pj, qj) - 1, 0); ej <= min(min(pj, qj), g.ey - 1); ej++)
                for (int ei = max(max(pi, qi) - 1, 0); ei <= min(min(pi, qi), g.ex - 1); ei++) {
                    const long e = ei + (long)g.ex * (ej + (long)g.ey * ek);
                    const int la = corner_id(pi - ei, pj - ej, pk - ek), lb = corner_id(qi - ei, qj - ej, qk - ek);
                    double v = cK * kf[e] * KE[(3 * la + c) * 24 + 3 * lb + d];
                    if (c == d) v += cM * mf[e] * M8[la * 8 + lb];
                    val += v;
                }
    }
    A[(size_t)i * n + j] = val;
}
void launch_dense_coarse(const Grid& g, const double* kf, const double* mf, double cK, double cM, const double* KE,
                         const double* M8, const uint8_t* mask, double* A, hipStream_t s) {
    const int n = (int)g.nd;
    TT_HIP(hipMemsetAsync(A, 0, (size_t)n * n * sizeof(double), s));
    hipLaunchKernelGGL(k_dense_coarse, dim3(nblocks((long)n * 81)), dim3(BS), 0, s, gargs(g), kf, mf, cK, cM, KE, M8,
                       mask, n, A);
    TT_HIP(hipGetLastError());
}

// ---- symmetric coarsest solve on the packed lower triangle: 64 x 64 tiles (I, J), I >= J, stored
// contiguously in row-major order, tile index I (I + 1) / 2 + J.  Half the bytes of the full matrix.
constexpr int ST = 64;
static inline int sym_tiles(int n) { return (n + ST - 1) / ST; }
long sym_packed_size(int n) {
    const long nt = sym_tiles(n);
    return nt * (nt + 1) / 2 * ST * ST;
}
// pack the lower triangle of the full symmetric matrix A (n x n) into tiles (zero padded)
__global__ void k_sym_pack(const double* __restrict__ A, int n, double* __restrict__ P) {
    const int I = blockIdx.y, J = blockIdx.x;
    if (J > I) return;
    double* T = P + ((size_t)I * (I + 1) / 2 + J) * ST * ST;
    for (int e = threadIdx.x; e < ST * ST; e += blockDim.x) {
        const int r = e / ST, c = e % ST, i = I * ST + r, j = J * ST + c;
        T[e] = (i < n && j < n) ? A[(size_t)i * n + j] : 0.0;
    }
}
void launch_sym_pack(const double* A, int n, double* P, hipStream_t s) {
    const int nt = sym_tiles(n);
    hipLaunchKernelGGL(k_sym_pack, dim3(nt, nt), dim3(256), 0, s, A, n, P);
    TT_HIP(hipGetLastError());
}
// per tile: row sums A_IJ x_J and (off the diagonal) column sums A_IJ^T x_I, written as FP64 partials.  Each thread
// holds 8 rows (tid / 32 + 8 k) x 2 columns of the tile in registers (16-byte loads, all in flight): its columns' sums go
// through LDS over the 8 row groups, its rows' over the 32 lanes of the half wave by halving exchanges (9 instead of
// 40 shuffles).  HBM bound: 68 MB at 4,131 dofs, see k_sym_sum.
__global__ __launch_bounds__(256) void k_sym_tiles(const double* __restrict__ P, const double* __restrict__ x, int n,
                                                   double* __restrict__ prow, double* __restrict__ pcol) {
    __shared__ double cs[8][ST];
    const int id = blockIdx.x;
    int I = (int)((sqrt(8.0 * id + 1.0) - 1.0) * 0.5);  // I (I + 1) / 2 <= id < (I + 1)(I + 2) / 2
    while ((I + 1) * (I + 2) / 2 <= id) I++;
    while (I * (I + 1) / 2 > id) I--;
    const int J = id - I * (I + 1) / 2;
    const double2* T2 = reinterpret_cast<const double2*>(P + (size_t)id * ST * ST);
    const int tid = threadIdx.x, rg = tid >> 5, c = 2 * (tid & 31);
    double2 v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = T2[tid + 256 * k];
    const int j = J * ST + c, i = I * ST + rg;
    const double x0 = j < n ? x[j] : 0.0, x1 = j + 1 < n ? x[j + 1] : 0.0;
    double xi[8], rs[8], c0 = 0.0, c1 = 0.0;
#pragma unroll
    for (int k = 0; k < 8; k++) xi[k] = i + 8 * k < n ? x[i + 8 * k] : 0.0;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        rs[k] = fma(v[k].x, x0, v[k].y * x1);
        c0 = fma(v[k].x, xi[k], c0);
        c1 = fma(v[k].y, xi[k], c1);
    }
    cs[rg][c] = c0;
    cs[rg][c + 1] = c1;
    // after the exchange over lane bit 4, 3, 2 a lane keeps 4, 2, 1 of its rows
    int row = rg;
#pragma unroll
    for (int b = 0; b < 3; b++) {
        const int h = 4 >> b, bit = 16 >> b;
        const bool up = (tid & bit) != 0;
        row += up ? 8 * h : 0;
#pragma unroll
        for (int m = 0; m < 4; m++)
            if (m < h) {
                const double keep = up ? rs[m + h] : rs[m], send = up ? rs[m] : rs[m + h];
                rs[m] = keep + __shfl_xor(send, bit, 64);
            }
    }
    rs[0] += __shfl_xor(rs[0], 2, 64);
    rs[0] += __shfl_xor(rs[0], 1, 64);
    if ((tid & 3) == 0) prow[(size_t)id * ST + row] = rs[0];
    __syncthreads();
    if (tid < ST) {
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < 8; q++) s += cs[q][tid];
        pcol[(size_t)id * ST + tid] = I == J ? 0.0 : s;
    }
}
// y_i = sum_{J <= I} prow(I, J) + sum_{K > I} pcol(K, I): one block per tile row I, 16 threads per output summing every
// 16th partial (their loads in flight together), combined in a fixed order
__global__ __launch_bounds__(1024) void k_sym_sum(const double* __restrict__ prow, const double* __restrict__ pcol,
                                                  int n, int nt, double* __restrict__ y) {
    __shared__ double red[16][ST];
    const int I = blockIdx.x, q = threadIdx.x >> 6, r = threadIdx.x & 63;
    double s = 0.0;
#pragma unroll 8
    for (int m = q; m < nt; m += 16) {  // m <= I: tile (I, m) rows; m > I: tile (m, I) columns
        const double* p = m <= I ? prow + ((size_t)I * (I + 1) / 2 + m) * ST : pcol + ((size_t)m * (m + 1) / 2 + I) * ST;
        s += p[r];
    }
    red[q][r] = s;
    __syncthreads();
    const int i = I * ST + threadIdx.x;
    if (threadIdx.x < ST && i < n) {
        double t = 0.0;
#pragma unroll
        for (int g = 0; g < 16; g++) t += red[g][threadIdx.x];
        y[i] = t;
    }
}
// y = A x with the full matrix, one wave per row: for small orders, where the matrix sits in L2 and the second launch of
// the packed form is what counts
__global__ __launch_bounds__(256) void k_dense_mv(const double* __restrict__ A, const double* __restrict__ x, int n,
                                                  double* __restrict__ y) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= n) return;
    const double* a = A + (size_t)row * n;
    double s = 0.0;
#pragma unroll 8
    for (int j = lane; j < n; j += 64) s = fma(a[j], x[j], s);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) y[row] = s;
}
void launch_sym_solve(const double* A, const double* P, const double* b, double* x, int n, double* prow, double* pcol,
                      hipStream_t s) {
    if (n <= kDenseMvMax) {
        hipLaunchKernelGGL(k_dense_mv, dim3((n + 3) / 4), dim3(256), 0, s, A, b, n, x);
        TT_HIP(hipGetLastError());
        return;
    }
    const int nt = sym_tiles(n);
    hipLaunchKernelGGL(k_sym_tiles, dim3(nt * (nt + 1) / 2), dim3(256), 0, s, P, b, n, prow, pcol);
    TT_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_sym_sum, dim3(nt), dim3(1024), 0, s, prow, pcol, n, nt, x);
    TT_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ reductions / Krylov
// Reductions over long vectors use at most RB blocks (grid-stride), so that the
// consumers of their partials (next kernel or host) sum few values.
constexpr int RB = 1024;
static inline int rb_blocks(long n) {
    int b = nblocks(n);
    return b > RB ? RB : (b < 1 ? 1 : b);
}

__global__ void k_dot(const double* __restrict__ a, const double* __restrict__ b, long n, double* part) {
    double acc[1] = {0.0};
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        acc[0] = fma(a[i], b[i], acc[0]);
    write_partials<1>(acc, part);
}
void launch_dot(const double* a, const double* b, long n, Reducer& red, int region, hipStream_t s) {
    const int nb = rb_blocks(n);
    hipLaunchKernelGGL(k_dot, dim3(nb), dim3(BS), 0, s, a, b, n, red.part(region));
    red.nblk[region] = nb;
    red.nv[region] = 1;
    TT_HIP(hipGetLastError());
}

__global__ void k_expand3(Expand3 e, long n) {
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
    for (int k = 0; k < e.nb; k++) {
        const double q = e.Q[(size_t)k * n + i];
        s0 = fma(e.c[0][k], q, s0);
        s1 = fma(e.c[1][k], q, s1);
        s2 = fma(e.c[2][k], q, s2);
    }
    e.out[0][i] = s0;
    if (e.nout > 1) e.out[1][i] = s1;
    if (e.nout > 2) e.out[2][i] = s2;
}
void launch_expand3(const Expand3& e, long n, hipStream_t s) {
    TT_CHECK(e.nb >= 1 && e.nb <= 64 && e.nout >= 1 && e.nout <= 3, -3, "launch_expand3: 1..64 vectors, 1..3 outputs");
    hipLaunchKernelGGL(k_expand3, dim3(nblocks(n)), dim3(BS), 0, s, e, n);
    TT_HIP(hipGetLastError());
}

__global__ void k_axpy_multi(Expand3 e, long n) {
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    double s0 = e.out[0][i];
#pragma unroll 4
    for (int k = 0; k < e.nb; k++) s0 = fma(e.c[0][k], e.Q[(size_t)k * n + i], s0);
    e.out[0][i] = s0;
}
void launch_axpy_multi(const Expand3& e, long n, hipStream_t s) {
    TT_CHECK(e.nb >= 1 && e.nb <= 64, -3, "launch_axpy_multi: 1..64 vectors");
    hipLaunchKernelGGL(k_axpy_multi, dim3(nblocks(n)), dim3(BS), 0, s, e, n);
    TT_HIP(hipGetLastError());
}

// Modified Gram-Schmidt in passes over groups of vectors.  One pass subtracts the current group (its coefficients from
// the dots that the previous pass left) and forms the dots of the new w with the next group, or, after the last, with
// its own group and itself.  With D_i = w.v_i at the group's start, the coefficients one after the other are
// h_i = D_i - sum_{j < i} h_j (v_j.v_i): those of subtracting v_0, v_1, ... in turn up to rounding (in exact arithmetic
// the same; D_i is taken before the group's own vectors are subtracted), with the stored dots of the group's vectors.
// Bound by memory: (2 + group + next group) vectors a pass, 30 us at 128x64x64 (7.8 TB/s, above the 6.5 of a copy: the last
// level of cache holds part of them), against a dot product, a host round trip and an update (5 vectors and ~28 us) per
// vector before: an Arnoldi step of 16 vectors takes 90 instead of 450 us.
constexpr int MG = kMgsGroup, MB = kMgsBlocks, MT = 512;
static_assert(MT / 64 == MG, "one wave sums one entry");
// entry q of the MB partial rows, summed by wave q (fixed order), into d[q]; entry MG by wave 0
__device__ __forceinline__ void mgs_sums(const double* __restrict__ part, double* d) {
    const int q = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int e = q; e <= MG; e += MG) {
        double x = 0.0;
#pragma unroll
        for (int b = 0; b < MB / 64; b++) x += part[(size_t)(lane + 64 * b) * (MG + 1) + e];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
        if (lane == 0) d[e] = x;
    }
    __syncthreads();
}
__global__ __launch_bounds__(MT) void k_mgs(double* __restrict__ w, const double* __restrict__ V, long n, int i0, int na,
                                            int nnext, const double* __restrict__ part_in,
                                            double* __restrict__ part_out, const double* __restrict__ G,
                                            double* __restrict__ h) {
    __shared__ double d[MG + 1], hs[MG], sh[16 * (MG + 1)];
    if (threadIdx.x < MG) hs[threadIdx.x] = 0.0;
    if (na > 0) {
        mgs_sums(part_in, d);
        if (threadIdx.x == 0)
            for (int i = 0; i < na; i++) {
                double x = d[i];
                for (int j = 0; j < i; j++) x = fma(-hs[j], G[(i0 + j) * kMgsMax + i0 + i], x);
                hs[i] = x;
                if (blockIdx.x == 0) h[i0 + i] = x;
            }
    }
    __syncthreads();
    const double* Va = V + (size_t)i0 * n;
    const double* Vb = Va + (size_t)na * n;
    double hq[MG], acc[MG + 1];
#pragma unroll
    for (int q = 0; q < MG; q++) hq[q] = hs[q];
#pragma unroll
    for (int q = 0; q <= MG; q++) acc[q] = 0.0;
    for (long i = blockIdx.x * (long)MT + threadIdx.x; i < n; i += (long)MB * MT) {
        double va[MG], vb[MG];
        double wi = w[i];
#pragma unroll
        for (int q = 0; q < MG; q++) va[q] = q < na ? Va[(size_t)q * n + i] : 0.0;
#pragma unroll
        for (int q = 0; q < MG; q++) vb[q] = q < nnext ? Vb[(size_t)q * n + i] : 0.0;
#pragma unroll
        for (int q = 0; q < MG; q++)
            if (q < na) wi = fma(-hq[q], va[q], wi);
        if (na > 0) w[i] = wi;
#pragma unroll
        for (int q = 0; q < MG; q++) acc[q] = fma(wi, nnext > 0 ? vb[q] : va[q], acc[q]);
        acc[MG] = fma(wi, wi, acc[MG]);
    }
    block_sum<MG + 1>(acc, sh);
    if (threadIdx.x == 0)
#pragma unroll
        for (int q = 0; q <= MG; q++) part_out[(size_t)blockIdx.x * (MG + 1) + q] = acc[q];
}
// w /= ||w||, h[k] = ||w||, and the dots of the new vector k with the earlier ones of its group (the last pass's)
__global__ __launch_bounds__(MT) void k_mgs_scale(double* __restrict__ w, long n, int k, const double* __restrict__ part,
                                                  double* __restrict__ G, double* __restrict__ h) {
    __shared__ double d[MG + 1];
    mgs_sums(part, d);
    const double nrm = sqrt(d[MG]), inv = nrm > 0.0 ? 1.0 / nrm : 1.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        h[k] = nrm;
        const int g0 = k / MG * MG;
        for (int i = g0; i < k; i++) G[i * kMgsMax + k] = d[i - g0] * inv;
    }
    for (long i = blockIdx.x * (long)MT + threadIdx.x; i < n; i += (long)MB * MT) w[i] *= inv;
}
void launch_mgs(double* w, const double* V, int k, long n, double* G, double* h, double* part, hipStream_t s) {
    TT_CHECK(k >= 1 && k < kMgsMax, -3, "launch_mgs: 1..31 vectors");
    double* pb[2] = {part, part + (size_t)MB * (MG + 1)};
    int cur = 0;
    hipLaunchKernelGGL(k_mgs, dim3(MB), dim3(MT), 0, s, w, V, n, 0, 0, std::min(MG, k), pb[1], pb[0], G, h);
    for (int i0 = 0; i0 < k; i0 += MG) {
        const int na = std::min(MG, k - i0), nn = std::min(MG, std::max(0, k - i0 - na));
        hipLaunchKernelGGL(k_mgs, dim3(MB), dim3(MT), 0, s, w, V, n, i0, na, nn, pb[cur], pb[cur ^ 1], G, h);
        cur ^= 1;
    }
    hipLaunchKernelGGL(k_mgs_scale, dim3(MB), dim3(MT), 0, s, w, n, k, pb[cur], G, h);
    TT_HIP(hipGetLastError());
}

template <int NQ>
__global__ void k_proj3(const double* __restrict__ Q, int k0, const double* __restrict__ a,
                        const double* __restrict__ b, const double* __restrict__ c, long n, double* part) {
    double acc[3 * NQ];
#pragma unroll
    for (int j = 0; j < 3 * NQ; j++) acc[j] = 0.0;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        const double ai = a[i], bi = b[i], ci = c[i];
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const double qi = Q[(size_t)(k0 + q) * n + i];
            acc[3 * q] = fma(qi, ai, acc[3 * q]);
            acc[3 * q + 1] = fma(qi, bi, acc[3 * q + 1]);
            acc[3 * q + 2] = fma(qi, ci, acc[3 * q + 2]);
        }
    }
    __shared__ double sh[(BS / 64) * 3 * NQ];
    block_sum<3 * NQ>(acc, sh);
    if (threadIdx.x == 0)
#pragma unroll
        for (int q = 0; q < NQ; q++)
            for (int j = 0; j < 3; j++) part[((size_t)(k0 + q) * RB + blockIdx.x) * 3 + j] = acc[3 * q + j];
}
int launch_proj3(const double* Q, int k0, int nq, const double* a, const double* b, const double* c, long n,
                 double* part, hipStream_t s) {
    const int nb = rb_blocks(n);
    switch (nq) {
#define TT_PROJ3(NQ) \
    case NQ: hipLaunchKernelGGL(k_proj3<NQ>, dim3(nb), dim3(BS), 0, s, Q, k0, a, b, c, n, part); break;
        TT_PROJ3(1) TT_PROJ3(2) TT_PROJ3(3) TT_PROJ3(4) TT_PROJ3(5) TT_PROJ3(6) TT_PROJ3(7) TT_PROJ3(8)
#undef TT_PROJ3
    default: throw Error{-3, "launch_proj3: 1..8 vectors per launch"};  // TT_ERR_INTERNAL
    }
    TT_HIP(hipGetLastError());
    return nb;
}

// partials of z.r and z.q_old (flexible CG, Polak-Ribiere form; see fcg_beta)
__global__ void k_fcg_dots(const double* __restrict__ z, const double* __restrict__ r, const double* __restrict__ q,
                           long n, double* part, int first) {
    double acc[2] = {0.0, 0.0};
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        acc[0] = fma(z[i], r[i], acc[0]);
        if (!first) acc[1] = fma(z[i], q[i], acc[1]);
    }
    write_partials<2>(acc, part);
}
void launch_fcg_dots(const double* z, const double* r, const double* q_old, long n, Reducer& red, bool first,
                     hipStream_t s) {
    const int nb = rb_blocks(n);
    hipLaunchKernelGGL(k_fcg_dots, dim3(nb), dim3(BS), 0, s, z, r, q_old, n, red.part(PB_DOTS), (int)first);
    red.nblk[PB_DOTS] = nb;
    red.nv[PB_DOTS] = 2;
    TT_HIP(hipGetLastError());
}

// Start (or restart) of a flexible-CG solve, from the partials of b.b and of r.r for the current
// x: the tolerance (rtol ||b||)^2, whether b = 0, and whether x already meets the tolerance.  The
// b.b total replaces the first partial of its region (which then counts one block): the host reads
// it back at every convergence look, and a copy of a few thousand partials takes a slower path
// (measured: ~20 us more per look for 21 KB than for 8 KB).
__global__ __launch_bounds__(BSR) void k_fcg_init(double* __restrict__ bb_part, int bb_nblk, const double* __restrict__ rr_part,
                           int rr_nblk, double rtol2, int reset_iters, double* scal, double* look) {
    double bb[1], rr[1];
    sum_partials<1>(bb_part, bb_nblk, bb);
    sum_partials<1>(rr_part, rr_nblk, rr);
    if (threadIdx.x == 0) {
        bb_part[0] = bb[0];
        look[Reducer::kLookBB] = bb[0];
        const double tol2 = rtol2 * bb[0];
        scal[SC_TOL2] = tol2;
        scal[SC_ZERO] = bb[0] == 0.0 ? 1.0 : 0.0;
        scal[SC_DONE] = (bb[0] == 0.0 || rr[0] <= tol2) ? 1.0 : 0.0;
        if (reset_iters) scal[SC_ITERS] = 0.0;
    }
}
void launch_fcg_init(Reducer& red, int bb_region, int rr_region, double rtol2, bool reset_iters, hipStream_t s) {
    hipLaunchKernelGGL(k_fcg_init, dim3(1), dim3(BSR), 0, s, red.part(bb_region), red.nblk[bb_region] * red.nv[bb_region],
                       red.part(rr_region), red.nblk[rr_region] * red.nv[rr_region], rtol2, reset_iters ? 1 : 0,
                       red.scal.p, red.look_dev);
    TT_HIP(hipGetLastError());
    red.nblk[bb_region] = 1;
    red.nv[bb_region] = 1;
}

// x += alpha p (x = 0 if b = 0); r -= alpha q; partials of r.r.  Every block forms alpha = gamma / (p.q) itself from the
// p.q partials, and checks the previous update's r.r (not on the first iteration of a (re)start): once that is
// <= (rtol ||b||)^2, SC_DONE is set and alpha is 0 for the rest of the solve, so x is frozen at the first iteration that
// met the tolerance; a frozen solve keeps x and r as they are.  Block 0 writes the scalars: what other blocks read of
// them gives the same decision before and after that write (SC_DONE is only ever set to what they find themselves).
// HBM bound: 6 vectors, 16 us at 128x64x64 (4.9 TB/s; with r_prev written as a 7th vector, which z.q_old makes unnecessary,
// and a one-block kernel for alpha before it: 17 + 4.7 us).
template <bool JAC>
__global__ __launch_bounds__(BS) void k_fcg_update(double* __restrict__ x, const double* __restrict__ p,
                                                   double* __restrict__ r, const double* __restrict__ q, long n,
                                                   const double* __restrict__ pq_part, int pq_nblk,
                                                   const double* __restrict__ rr_old, int rr_nblk, double* scal,
                                                   double* part, double* look, int first,
                                                   const double* __restrict__ dinv, double* dots) {
    const long i0 = blockIdx.x * (long)blockDim.x + threadIdx.x, st = (long)gridDim.x * blockDim.x;
    // the first values are in flight while the partials are summed
    double x0 = 0.0, p0 = 0.0, r0 = 0.0, q0 = 0.0;
    if (i0 < n) {
        x0 = x[i0];
        p0 = p[i0];
        r0 = r[i0];
        q0 = q[i0];
    }
    const double s_zero = scal[SC_ZERO], s_done = scal[SC_DONE], tol2 = scal[SC_TOL2], gam = scal[SC_GAMMA];
    double pq[1], rr[1] = {0.0};
    sum_partials<1>(pq_part, pq_nblk, pq);
    if (!first) sum_partials<1>(rr_old, rr_nblk, rr);
    const bool zero = s_zero != 0.0, done = s_done != 0.0 || (!first && rr[0] <= tol2);
    const double al = done ? 0.0 : gam / pq[0];
    constexpr int NA = JAC ? 3 : 1;
    double acc[NA];
#pragma unroll
    for (int k = 0; k < NA; k++) acc[k] = 0.0;
    for (long i = i0; i < n; i += st) {
        if (i != i0) {
            x0 = x[i];
            p0 = p[i];
            r0 = r[i];
            q0 = q[i];
        }
        if (zero) x[i] = 0.0;
        else if (!done) x[i] = fma(al, p0, x0);
        const double rn = done ? r0 : fma(-al, q0, r0);
        if (!done) r[i] = rn;
        acc[0] = fma(rn, rn, acc[0]);
        if constexpr (JAC) {  // (q0 is the next direction's q_old)
            const double z = dinv[i] * rn;
            acc[1] = fma(z, rn, acc[1]);
            acc[2] = fma(z, q0, acc[2]);
        }
    }
    __shared__ double sh[16 * NA];
    block_sum<NA>(acc, sh);
    if (threadIdx.x == 0) {  // the partial for the next update, and its copy for the host's look
        part[blockIdx.x] = acc[0];
        look[blockIdx.x] = acc[0];
        if constexpr (JAC) {
            dots[2 * blockIdx.x] = acc[1];
            dots[2 * blockIdx.x + 1] = acc[2];
        }
        if (blockIdx.x == 0) {
            const double it = scal[SC_ITERS] + (done ? 0.0 : 1.0);
            scal[SC_DONE] = done ? 1.0 : 0.0;
            scal[SC_ALPHA] = al;
            scal[SC_GAMMA_OLD] = gam;
            scal[SC_ITERS] = it;
            look[gridDim.x] = it;
        }
    }
}
void launch_fcg_update(double* x, const double* p, double* r, const double* q, long n, Reducer& red, bool first,
                       bool odd, hipStream_t s, const double* dinv) {
    const int nb = rb_blocks(n), now = rr_region(odd), old = rr_region(!odd);
    TT_CHECK(nb < Reducer::kLookBB, -3, "look buffer too small");
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(nb), dim3(BS), 0, s, x, p, r, q, n, red.part(PB_PQ), red.nblk[PB_PQ],
                           red.part(old), red.nblk[old], red.scal.p, red.part(now), red.look_dev, first ? 1 : 0, dinv,
                           red.part(PB_DOTS));
    };
    if (dinv) {
        launch(k_fcg_update<true>);
        red.nblk[PB_DOTS] = nb;
        red.nv[PB_DOTS] = 2;
    } else {
        launch(k_fcg_update<false>);
    }
    red.nblk[now] = nb;
    red.nv[now] = 1;
    TT_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ PDE filter operator (PDEFilter.cc)
// On the node grid of a box the Helmholtz matrix is a sum of products of 1-D matrices (stiffness K = [-1 c -1] / h, mass
// M = [1 2c 1] h / 6 per direction, c = the 1 or 2 elements at the node), R^2 (Kx My Mz + Mx Ky Mz + Mx My Kz) +
// Mx My Mz.  A block owns BX x BY node columns (32 x 8, narrower where the grid is) and marches up its planes: a plane (with one halo node) is staged in LDS,
// each thread forms A = My Mx u and B = (R^2 (Kx My + Mx Ky) + Mx My) u of its column from the 9 neighbours, and the
// row sum is Mz B + R^2 Kz A over three planes.  The staged value is the solution (the residual) or the CG direction
// formed on the fly.  At 128x64x64 a CG iteration's two kernels (this one and k_fcg_update) replace seven (48 us:
// Jacobi, dots, beta, direction, an apply that gathered 64 products per node, alpha, update).
// A cross-section of up to 8 x 8 nodes takes S = 4 or 16 parts of a block's planes side by side (strands, as the operator's
// columns).  Whole filter calls on device arrays, us, the node-by-node operator of seven kernels an iteration that the march
// replaced, 32 x 8 tiles alone, and tiles by the grid: 1x1x20000 elements 696 -> 963 -> 585, 3x3x30000 1173 -> 1384 -> 705,
// 3x30000x3 1107 -> 1498 -> 695, 1x500x500 1182 -> 1651 -> 733, 1x1000x1000 3247 -> 5084 -> 1501 (129 x 65 x 65 nodes: the
// same tiles as before).
template <int LBX, int LBY>
struct FilterTile {
    static constexpr int BX = 1 << LBX, BY = 1 << LBY, S = 256 >> (LBX + LBY), HX = BX + 2, BOX = HX * (BY + 2),
                         Q = (S * BOX + 255) / 256;  // staged nodes per strand and per thread
};
template <bool CG, int LBX, int LBY>  // CG: u = p = D^-1 r + beta p_old (written), y = q = A p, partials of p.q; else y = rhs - A u
__global__ __launch_bounds__(256) void k_filter_op(GridArgs g, FilterOp f, int tx, int ty, int tz,
                                                   const double* __restrict__ a0, const double* __restrict__ dinv,
                                                   const double* __restrict__ a1, double* __restrict__ pnew,
                                                   double* __restrict__ y, double* part0, double* part1, double* part2,
                                                   const double* dots, int dots_nblk, double* scal, int first) {
    typedef FilterTile<LBX, LBY> F;
    constexpr int S = F::S, FHX = F::HX, Q = F::Q;
    __shared__ double su[2][S * F::BOX];
    const int tid = threadIdx.x, lx = tid & (F::BX - 1), ly = (tid >> LBX) & (F::BY - 1);
    const int tile = blockIdx.x, tzi = tile / (tx * ty), tr = tile - tzi * tx * ty, tyi = tr / tx, txi = tr - tyi * tx;
    const int i0 = txi * F::BX, j0 = tyi * F::BY;
    const int k0 = (int)((long)tzi * g.nz / tz), nk = (int)((long)(tzi + 1) * g.nz / tz) - k0;
    // a strand's planes, and the thread's: koff above the march's, below kend
    const int np = (nk + S - 1) / S, koff = (S > 1 ? tid >> (LBX + LBY) : 0) * np, kend = k0 + min(koff + np, nk);
    const int i = i0 + lx, j = j0 + ly;
    const bool own = i < g.nx && j < g.ny;
    double beta = 0.0;
    if constexpr (CG) beta = fcg_beta(dots, dots_nblk, scal, first);
    // 1-D rows of the thread's node (a neighbour outside the grid has weight 0 at a valid index)
    auto row = [](int n, int nn, double h, double (&m)[3], double (&k)[3]) {
        const double l = n > 0 ? 1.0 : 0.0, r = n < nn - 1 ? 1.0 : 0.0, c = l + r;
        m[0] = l * (h / 6.0); m[1] = c * (h / 3.0); m[2] = r * (h / 6.0);
        k[0] = -l / h; k[1] = c / h; k[2] = -r / h;
    };
    double mx[3], kx[3], my[3], ky[3];
    row(i, g.nx, f.h[0], mx, kx);
    row(j, g.ny, f.h[1], my, ky);
    // staging: Q of the box nodes per thread
    int so[Q], sk[Q];
    bool sv[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int v = tid + q * 256, st = S > 1 ? min(v / F::BOX, S - 1) : 0, w = v - st * F::BOX, sy = w / FHX,
                  sx = w - sy * FHX;
        sv[q] = v < S * F::BOX;
        sk[q] = st * np;
        so[q] = min(max(i0 - 1 + sx, 0), g.nx - 1) + g.nx * min(max(j0 - 1 + sy, 0), g.ny - 1);
    }
    const int plane = g.nx * g.ny;
    double v0[Q], v1[Q], v2[Q];
    auto load = [&](int k) {
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const size_t b = (size_t)min(max(S > 1 ? k + sk[q] : k, 0), g.nz - 1) * plane;
            v0[q] = a0[b + so[q]];
            if constexpr (CG) {
                v1[q] = dinv[b + so[q]];
                v2[q] = first ? 0.0 : a1[b + so[q]];
            }
        }
    };
    auto commit = [&](int b) {
#pragma unroll
        for (int q = 0; q < Q; q++) {
            double x = v0[q];
            if constexpr (CG) {
                x = v1[q] * v0[q];
                if (!first) x = fma(beta, v2[q], x);
            }
            if (sv[q]) su[b][tid + q * 256] = x;
        }
    };
    double A[3] = {0, 0, 0}, B[3] = {0, 0, 0}, uo[2] = {0, 0}, acc[3] = {0, 0, 0};
    load(k0 - 1);
    commit(0);
    __syncthreads();
    for (int k = k0 - 1; k <= k0 + np; k++) {  // plane k is staged in su[(k - k0 + 1) & 1]
        const int sb = (k - k0 + 1) & 1;
        if (k < k0 + np) load(k + 1);
        double As = 0.0, Bs = 0.0;
        const double* u = &su[sb][(S > 1 ? (tid >> (LBX + LBY)) * F::BOX : 0) + ly * FHX + lx];
#pragma unroll
        for (int r = 0; r < 3; r++) {
            const double ul = u[r * FHX], uc = u[r * FHX + 1], ur = u[r * FHX + 2];
            const double um = fma(mx[0], ul, fma(mx[1], uc, mx[2] * ur)), uk = fma(kx[0], ul, fma(kx[1], uc, kx[2] * ur));
            As = fma(my[r], um, As);
            Bs = fma(my[r], fma(f.R2, uk, um), Bs);
            Bs = fma(f.R2 * ky[r], um, Bs);
        }
        const double un = u[FHX + 1];
        A[0] = A[1]; A[1] = A[2]; A[2] = As;
        B[0] = B[1]; B[1] = B[2]; B[2] = Bs;
        const int kk = k - 1 + koff;  // the plane whose three neighbours are now known
        if (k > k0 && kk < kend && own) {
            double mz[3], kz[3];
            row(kk, g.nz, f.h[2], mz, kz);
            double s = 0.0;
#pragma unroll
            for (int d = 0; d < 3; d++) s = fma(mz[d], B[d], fma(f.R2 * kz[d], A[d], s));
            const size_t n = (size_t)kk * plane + i + (size_t)g.nx * j;
            if constexpr (CG) {
                y[n] = s;
                pnew[n] = uo[0];
                acc[0] = fma(uo[0], s, acc[0]);
            } else {
                const double b = a1[n], r = b - s;
                y[n] = r;
                acc[0] = fma(r, r, acc[0]);
                acc[1] = fma(dinv[n] * r, r, acc[1]);
                acc[2] = fma(b, b, acc[2]);
            }
        }
        uo[0] = un;
        if (k < k0 + np) commit(sb ^ 1);
        __syncthreads();
    }
    __shared__ double sh[16 * 3];
    block_sum<3>(acc, sh);
    if (tid == 0) {
        part0[tile] = acc[0];
        if constexpr (!CG) {
            part1[2 * tile] = acc[1];
            part1[2 * tile + 1] = 0.0;
            if (part2) part2[tile] = acc[2];
        }
    }
}
// tiles: about 4 blocks per CU, at least one plane (of each strand)
struct FilterPlan {
    int lbx, lby, tx, ty, tz;
    int blocks() const { return tx * ty * tz; }
};
static inline FilterPlan filter_plan(const Grid& g) {
    FilterPlan p{5, 3, 0, 0, 0};
    while (p.lbx > 2 && (1 << (p.lbx - 1)) >= g.nx) p.lbx--;
    p.lby = 8 - p.lbx;
    if (g.nx <= 8 && g.ny <= 8) p.lbx = p.lby = g.nx <= 4 && g.ny <= 4 ? 2 : 3;
    const int s = 256 >> (p.lbx + p.lby);
    p.tx = (g.nx + (1 << p.lbx) - 1) >> p.lbx;
    p.ty = (g.ny + (1 << p.lby) - 1) >> p.lby;
    p.tz = std::min((g.nz + s - 1) / s, std::max(1, 1024 / (p.tx * p.ty)));
    return p;
}
long filter_blocks(const Grid& g) { return filter_plan(g).blocks(); }
template <bool CG, class... Args>
static void filter_op(const Grid& g, const FilterPlan& p, hipStream_t s, const FilterOp& f, Args... args) {
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(p.blocks()), dim3(256), 0, s, gargs(g), f, p.tx, p.ty, p.tz, args...);
    };
    if (p.lbx + p.lby < 8) p.lbx == 2 ? launch(k_filter_op<CG, 2, 2>) : launch(k_filter_op<CG, 3, 3>);
    else if (p.lbx == 5) launch(k_filter_op<CG, 5, 3>);
    else if (p.lbx == 4) launch(k_filter_op<CG, 4, 4>);
    else if (p.lbx == 3) launch(k_filter_op<CG, 3, 5>);
    else launch(k_filter_op<CG, 2, 6>);
    TT_HIP(hipGetLastError());
}
void launch_filter_residual(const Grid& g, const FilterOp& f, const double* U, const double* rhs, const double* dinv,
                            double* r, Reducer& red, bool bb, hipStream_t s) {
    const FilterPlan p = filter_plan(g);
    const int nb = p.blocks();
    TT_CHECK(nb <= red.maxblocks, -3, "reducer too small");
    filter_op<false>(g, p, s, f, U, dinv, rhs, (double*)nullptr, r, red.part(PB_MISC2), red.part(PB_DOTS),
                     bb ? red.part(PB_MISC) : (double*)nullptr, (const double*)nullptr, 0, (double*)nullptr, 0);
    for (int region : {(int)PB_MISC2, (int)PB_DOTS, (int)PB_MISC})
        if (region != PB_MISC || bb) {
            red.nblk[region] = nb;
            red.nv[region] = region == PB_DOTS ? 2 : 1;
        }
}
void launch_filter_direction(const Grid& g, const FilterOp& f, const double* r, const double* dinv, const double* p_old,
                             double* p_new, double* q, Reducer& red, bool first, hipStream_t s) {
    const FilterPlan p = filter_plan(g);
    const int nb = p.blocks();
    TT_CHECK(nb <= red.maxblocks, -3, "reducer too small");
    filter_op<true>(g, p, s, f, r, dinv, p_old, p_new, q, red.part(PB_PQ), (double*)nullptr, (double*)nullptr,
                    (const double*)red.part(PB_DOTS), red.nblk[PB_DOTS], red.scal.p, first ? 1 : 0);
    red.nblk[PB_PQ] = nb;
    red.nv[PB_PQ] = 1;
}

__global__ void k_jacobi(const double* __restrict__ dinv, const double* __restrict__ r, double* __restrict__ z,
                         long n) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) z[i] = dinv[i] * r[i];
}
void launch_jacobi(const double* dinv, const double* r, double* z, long n, hipStream_t s) {
    hipLaunchKernelGGL(k_jacobi, dim3(nblocks(n)), dim3(BS), 0, s, dinv, r, z, n);
    TT_HIP(hipGetLastError());
}

// power iteration helper: x = dinv.Ax, partials of ||x||^2 in PB_MISC
template <typename T>
__global__ void k_norm_power(const T* __restrict__ Ax, const T* __restrict__ dinv, T* __restrict__ x, long n,
                             double* part) {
    double acc[1] = {0.0};
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        const T v = dinv[i] * Ax[i];
        x[i] = v;
        acc[0] += (double)v * (double)v;
    }
    write_partials<1>(acc, part);
}
void launch_norm_power(const void* Ax, const void* dinv, void* x, long n, Reducer& red, bool fp64, hipStream_t s) {
    const int nb = rb_blocks(n);
    if (fp64)
        hipLaunchKernelGGL(k_norm_power<double>, dim3(nb), dim3(BS), 0, s, (const double*)Ax, (const double*)dinv,
                           (double*)x, n, red.part(PB_MISC));
    else
        hipLaunchKernelGGL(k_norm_power<float>, dim3(nb), dim3(BS), 0, s, (const float*)Ax, (const float*)dinv,
                           (float*)x, n, red.part(PB_MISC));
    red.nblk[PB_MISC] = nb;
    red.nv[PB_MISC] = 1;
    TT_HIP(hipGetLastError());
}

// x /= ||x|| with ||x||^2 summed from the partials of k_norm_power
template <typename T>
__global__ void k_scale_by_norm(T* x, long n, const double* part, int nblk) {
    double s[1];
    sum_partials<1>(part, nblk, s);
    const double inv = 1.0 / sqrt(s[0]);
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        x[i] = (T)((double)x[i] * inv);
}
void launch_scale_by_norm(void* x, long n, Reducer& red, bool fp64, hipStream_t s) {
    const int nb = rb_blocks(n);
    if (fp64)
        hipLaunchKernelGGL(k_scale_by_norm<double>, dim3(nb), dim3(BS), 0, s, (double*)x, n, red.part(PB_MISC),
                           red.nblk[PB_MISC]);
    else
        hipLaunchKernelGGL(k_scale_by_norm<float>, dim3(nb), dim3(BS), 0, s, (float*)x, n, red.part(PB_MISC),
                           red.nblk[PB_MISC]);
    TT_HIP(hipGetLastError());
}

__global__ void k_scale(double* x, long n, double a) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) x[i] *= a;
}
void launch_scale(double* x, long n, double a, hipStream_t s) {
    hipLaunchKernelGGL(k_scale, dim3(nblocks(n)), dim3(BS), 0, s, x, n, a);
    TT_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ Newmark / adjoint vector kernels
// corrector (LinearElasticity.cc:1363-1375): c = a[0..5].  The acceleration history of the new state
// is shifted in the same pass: hout[0] = a, hout[j] = hin[j - 1] (j < nh), vectors n apart.  With gout,
// the next step's initial guess sum_k gc.c[k] w_k over w = (un, vn, an, a, hin[0], hin[1]) is written as
// well, term by term in the order k_extrapolate sums the same vectors (bit-identical results).
struct GuessCoef {
    double c[6];
    int m;
};
__global__ void k_newmark_update(const double* u, const double* __restrict__ v,
                                 const double* __restrict__ a, const double* __restrict__ un, double* __restrict__ vn,
                                 double* __restrict__ an, double a0, double a1, double a2, double a3, double a4,
                                 double a5, long n, const double* __restrict__ hin, double* __restrict__ hout, int nh,
                                 GuessCoef gc, double* gout) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double ai = a[i];
    if (nh > 0) hout[i] = ai;
    for (int j = 1; j < nh; j++) hout[j * n + i] = hin[(j - 1) * n + i];
    const double uni = un[i];
    const double du = uni - u[i];
    double vv = 0.0;
    vv += a0 * v[i];
    vv += a1 * ai;
    vv += a2 * du;
    double aa = 0.0;
    aa += -a3 * v[i];
    aa += -a4 * ai;
    aa += a5 * du;
    vn[i] = vv;
    an[i] = aa;
    if (gout) {  // the next step's guess (gout may be this step's input u: u[i] is already read)
        double s = gc.c[0] * uni;
        if (gc.m > 1) s = fma(gc.c[1], vv, s);
        if (gc.m > 2) s = fma(gc.c[2], aa, s);
        if (gc.m > 3) s = fma(gc.c[3], ai, s);
        if (gc.m > 4) s = fma(gc.c[4], hin[i], s);
        if (gc.m > 5) s = fma(gc.c[5], hin[n + i], s);
        gout[i] = s;
    }
}
void launch_newmark_update(const double* u, const double* v, const double* a, const double* un, double* vn,
                           double* an, const double* c, long n, const double* hin, double* hout, int nh,
                           hipStream_t s, const Extrap* next, double* gout) {
    GuessCoef gc{};
    if (next) {
        TT_CHECK(next->m >= 1 && next->m <= 6 && nh >= 3, -3, "launch_newmark_update: guess of 1..6 terms");
        for (int k = 0; k < next->m; k++) gc.c[k] = next->c[k];
        gc.m = next->m;
    }
    hipLaunchKernelGGL(k_newmark_update, dim3(nblocks(n)), dim3(BS), 0, s, u, v, a, un, vn, an, c[0], c[1], c[2],
                       c[3], c[4], c[5], n, hin, hout, nh, gc, next ? gout : (double*)nullptr);
    TT_HIP(hipGetLastError());
}

// Adjoint step combination (LinearElasticity.cc:864-925).  coef = {a0..a5, dalpha, dbeta}.
// Kl = N K N lambda_{t+1}, Ml = N M N lambda_{t+1}; B1 = a5 M + a2 C, B2 = a3 M - a0 C, B3 = a4 M - a1 C.
// rhs = N.(-R1): the SPD form of the reference's solve with A = -(K + a2 C + a5 M).
struct AdjCoef {
    double a[6], al, be;
};
__global__ void k_adjoint_combine(const double* __restrict__ Kl, const double* __restrict__ Ml,
                                  const double* __restrict__ hdu, const double* __restrict__ hddu,
                                  const double* __restrict__ hdddu, const double* __restrict__ mun,
                                  const double* __restrict__ nun, const uint8_t* __restrict__ mask, AdjCoef c,
                                  int terminal, double* __restrict__ mu, double* __restrict__ nu,
                                  double* __restrict__ rhs, long nd) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= nd) return;
    const double* a = c.a;
    double m, v, r;
    if (terminal) {
        m = -hddu[i];
        v = -hdddu[i];
        r = hdu[i];
        r += -a[2] * m;
        r += -a[5] * v;
        r = -r;
    } else {
        const double kl = Kl[i], ml = Ml[i];
        const double b1 = (a[5] + a[2] * c.al) * ml + a[2] * c.be * kl;
        const double b2 = (a[3] - a[0] * c.al) * ml - a[0] * c.be * kl;
        const double b3 = (a[4] - a[1] * c.al) * ml - a[1] * c.be * kl;
        double mm = hddu[i];
        mm += b2;
        mm += -a[0] * mun[i];
        mm += a[3] * nun[i];
        double vv = hdddu[i];
        vv += b3;
        vv += a[4] * nun[i];
        r = hdu[i];
        r += b1;
        r += a[2] * mun[i];
        r += a[5] * nun[i];
        r = -r;
        m = -mm;
        v = -vv;
        r += a[2] * m;
        r += a[5] * v;
    }
    mu[i] = m;
    nu[i] = v;
    const bool clamped = (mask[i / 3] >> (i % 3)) & 1;
    rhs[i] = clamped ? 0.0 : -r;
}
void launch_adjoint_combine(const double* Kl, const double* Ml, const double* hdu, const double* hddu,
                            const double* hdddu, const double* mun, const double* nun, const uint8_t* mask,
                            const double* coef, bool terminal, double* mu, double* nu, double* rhs, long nn,
                            hipStream_t s) {
    AdjCoef c;
    for (int k = 0; k < 6; k++) c.a[k] = coef[k];
    c.al = coef[6];
    c.be = coef[7];
    long nd = 3 * nn;
    hipLaunchKernelGGL(k_adjoint_combine, dim3(nblocks(nd)), dim3(BS), 0, s, Kl, Ml, hdu, hddu, hdddu, mun, nun, mask,
                       c, (int)terminal, mu, nu, rhs, nd);
    TT_HIP(hipGetLastError());
}

// t = 0 adjoint right-hand side (LinearElasticity.cc:753-776): R3 = N.-(HDDDU + B3 l1 - a1 mu1 + a4 nu1)
__global__ void k_adjoint0_rhs(const double* __restrict__ Kl, const double* __restrict__ Ml,
                               const double* __restrict__ hdddu, const double* __restrict__ mun,
                               const double* __restrict__ nun, const uint8_t* __restrict__ mask, AdjCoef c,
                               double* __restrict__ rhs, long nd) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= nd) return;
    const double* a = c.a;
    const double b3 = (a[4] - a[1] * c.al) * Ml[i] - a[1] * c.be * Kl[i];
    double r = hdddu[i];
    r += b3;
    r += -a[1] * mun[i];
    r += a[4] * nun[i];
    const bool clamped = (mask[i / 3] >> (i % 3)) & 1;
    rhs[i] = clamped ? 0.0 : -r;
}
void launch_adjoint0_rhs(const double* Kl, const double* Ml, const double* hdddu, const double* mun,
                         const double* nun, const uint8_t* mask, const double* coef, double* rhs, long nn,
                         hipStream_t s) {
    AdjCoef c;
    for (int k = 0; k < 6; k++) c.a[k] = coef[k];
    c.al = coef[6];
    c.be = coef[7];
    long nd = 3 * nn;
    hipLaunchKernelGGL(k_adjoint0_rhs, dim3(nblocks(nd)), dim3(BS), 0, s, Kl, Ml, hdddu, mun, nun, mask, c, rhs, nd);
    TT_HIP(hipGetLastError());
}

// objectives 0..2: d/du of sum_e P_e dt/2 sum_k w_k^2 = dt * w_d * (sum of P over elements at the node)
__global__ void k_hdiag(const double* __restrict__ w, const double* __restrict__ cnt, double dt, double* __restrict__ h,
                        long nd) {
    long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < nd) h[i] = dt * w[i] * cnt[i / 3];
}
void launch_hdiag(const double* w, const double* cnt, double dt, double* h, long nn, hipStream_t s) {
    hipLaunchKernelGGL(k_hdiag, dim3(nblocks(3 * nn)), dim3(BS), 0, s, w, cnt, dt, h, 3 * nn);
    TT_HIP(hipGetLastError());
}
__global__ void k_region_count(GridArgs g, const double* __restrict__ P, double* __restrict__ cnt) {
    const long n = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (n >= (long)g.nx * g.ny * g.nz) return;
    const int i = n % g.nx, j = (n / g.nx) % g.ny, k = n / ((long)g.nx * g.ny);
    double s = 0.0;
    for (int ez = 0; ez < 2; ez++)
        for (int ey = 0; ey < 2; ey++)
            for (int ex = 0; ex < 2; ex++) {
                const int ei = i - 1 + ex, ej = j - 1 + ey, ek = k - 1 + ez;
                if (ei < 0 || ej < 0 || ek < 0 || ei >= g.ex || ej >= g.ey || ek >= g.ez) continue;
                s += P[ei + (long)g.ex * (ej + (long)g.ey * ek)];
            }
    cnt[n] = s;
}
void launch_region_count(const Grid& g, const double* P, double* cnt, hipStream_t s) {
    hipLaunchKernelGGL(k_region_count, dim3(nblocks(g.nn)), dim3(BS), 0, s, gargs(g), P, cnt);
    TT_HIP(hipGetLastError());
}

}  // namespace tt
