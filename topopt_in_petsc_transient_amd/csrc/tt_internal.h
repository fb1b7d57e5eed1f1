// Internal declarations of the MI355X transient-elasticity library.
//
// Layout in HBM (natural ordering of the reference's single-rank DMDA):
//   node  n = i + nx*(j + ny*k)      vectors: 3 dofs per node, interleaved (3n+c)
//   elem  e = i + ex*(j + ey*k)      per-element coefficients kfac/mfac
// Each multigrid level l holds its own element coefficients, Dirichlet mask
// (one byte per node, bit c set when dof c is clamped), inverse diagonal and
// vectors.  Precision of level vectors is FP64 in the FP64 mode and FP32 in
// the mixed mode; coarse-level coefficients are BF16 in the mixed mode.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>
#include <vector>

namespace tt {

typedef uint16_t bf16_t;

// ------------------------------------------------------------------ errors
struct Error {
    int code;
    std::string msg;
};

#define TT_HIP(call)                                                                            \
    do {                                                                                        \
        hipError_t e_ = (call);                                                                 \
        if (e_ != hipSuccess)                                                                   \
            throw ::tt::Error{-2, std::string("HIP error ") + hipGetErrorString(e_) + " at " +   \
                                      __FILE__ + ":" + std::to_string(__LINE__)};               \
    } while (0)

#define TT_CHECK(cond, code, msg)                      \
    do {                                               \
        if (!(cond)) throw ::tt::Error{(code), (msg)}; \
    } while (0)

// ------------------------------------------------------------------ device buffers
template <typename T>
struct DBuf {
    T* p = nullptr;
    size_t n = 0;
    DBuf() = default;
    explicit DBuf(size_t n_) { alloc(n_); }
    DBuf(const DBuf&) = delete;
    DBuf& operator=(const DBuf&) = delete;
    DBuf(DBuf&& o) noexcept : p(o.p), n(o.n) { o.p = nullptr; o.n = 0; }
    DBuf& operator=(DBuf&& o) noexcept {
        if (this != &o) { release(); p = o.p; n = o.n; o.p = nullptr; o.n = 0; }
        return *this;
    }
    ~DBuf() { release(); }
    void alloc(size_t n_) {
        release();
        n = n_;
        if (n) TT_HIP(hipMalloc((void**)&p, sizeof(T) * n));
    }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    T* get() const { return p; }
};

// message of a failed call made without a context (tt_last_error(NULL) returns it)
void set_contextless_error(const std::string& msg);

// ------------------------------------------------------------------ grid
struct Grid {
    int ex, ey, ez;  // elements
    int nx, ny, nz;  // nodes
    long nel, nn, nd;
    double hx, hy, hz;
};

inline Grid make_grid(int ex, int ey, int ez, double lx, double ly, double lz) {
    Grid g;
    g.ex = ex; g.ey = ey; g.ez = ez;
    g.nx = ex + 1; g.ny = ey + 1; g.nz = ez + 1;
    g.nel = (long)ex * ey * ez;
    g.nn = (long)g.nx * g.ny * g.nz;
    g.nd = 3 * g.nn;
    g.hx = lx / ex; g.hy = ly / ey; g.hz = lz / ez;
    return g;
}

// ------------------------------------------------------------------ host element matrices
void hex8_stiffness(double hx, double hy, double hz, double nu, double* ke);  // 24x24, E = 1
void hex8_mass(double hx, double hy, double hz, double* m8);                 // 8x8 scalar, density 1
void hex8_helmholtz(double hx, double hy, double hz, double R, double* kf);  // 8x8, R^2 Lap + mass

// The element matrices in the element's symmetry-adapted basis (mode bits x, y, z of the sums and differences of the
// corner values; see tt_apply_cols.inc): the stiffness matrix's blocks, upper triangles, and the mass matrix's
// diagonal by the number of odd directions.
template <typename T>
struct ModeConst {
    T n[6];     // ux100, uy010, uz001
    T q[3][3];  // (uy110, uz101), (ux110, uz011), (ux101, uy011)
    T s[3][3];  // (ux010, uy100), (ux001, uz100), (uy001, uz010)
    T t[6];     // ux011, uy101, uz110
    T d[3];     // ux111, uy111, uz111
    T m[4];
};
void hex8_modes(const double* ke, const double* m8, ModeConst<double>& mc);
// the same in device memory, in both precisions
void upload_modes(const double* ke, const double* m8, DBuf<ModeConst<double>>& d64, DBuf<ModeConst<float>>& d32);
// The tile split of one grid for the column kernels (tt_apply_cols.inc): columns of elements per tile row
// (bx + 1) and owned node columns per tile in x and y; tiles (the nz node planes are split evenly over tz).  cx = 0: a
// small grid, for the one-shot kernel (tt_apply_box.inc), whose tiles are 4 x 4 x 4 nodes.
struct ColTile {
    int cx, bx, by;
    int tx, ty, tz;
};
struct ColPlan : ColTile {
    int strands = 1;  // parts of a block's planes that march side by side (a rod's tile: its whole cross-section)
    int ntiles() const { return tx * ty * tz; }
    // blocks of a launch (column kernel: rounded up to a multiple of 8 for the XCD-aware tile order)
    int blocks() const { return cx ? 8 * ((ntiles() + 7) / 8) : ntiles(); }
};
ColPlan make_col_plan(const Grid& g, bool fp64);
// Per tile of a split: 1 if the tile's staged node box (one halo layer) holds a node with a nonzero mask.
void col_bc_flags(const Grid& g, const ColPlan& p, const std::vector<uint8_t>& mask, std::vector<uint8_t>& f);
struct ColSplit {
    ColPlan plan;
    const uint8_t* bc;  // the flags, in device memory
};
struct ColSplitStore {  // the splits of one grid, by precision, with their flags
    ColSplit s32{}, s64{};
    DBuf<uint8_t> flags[2];
    void build(const Grid& g, const std::vector<uint8_t>& mask);
};

// ------------------------------------------------------------------ reductions
// Deterministic device reductions without fences or atomics: a reducing kernel
// writes one partial per block into a partial buffer; the next kernel on the
// stream (or the host) sums the partials in block order.  Kernel boundaries
// give the visibility, so no block pays a device-scope fence (which on a
// multi-XCD GPU means an L2 write-back).
enum { PB_DOTS = 0, PB_PQ, PB_RR, PB_RR2, PB_MISC, PB_MISC2, PB_COUNT };
struct Reducer {
    DBuf<double> partials;   // PB_COUNT regions of [maxblocks * 4]
    DBuf<double> scal;       // device scalars (see SC_* indices)
    double* host = nullptr;  // pinned mirror of scal
    double* hpart = nullptr; // pinned host copy of one partial region
    // Host memory the kernels store into directly (pinned, mapped, coherent), so that the flexible-CG
    // convergence look needs no copy: [0, nb) the r.r partials of the last k_fcg_update, [nb] the
    // iterations that moved x; [kLookBB] the b.b of the solve (k_fcg_init).
    static constexpr int kLookBB = 1100;
    double* look = nullptr;
    double* look_dev = nullptr;  // the same memory as the kernels address it
    int maxblocks = 0;
    int nblk[PB_COUNT] = {};  // blocks that wrote each region
    int nv[PB_COUNT] = {};
    void init(int maxb);
    double* part(int region) const { return partials.p + (size_t)region * maxblocks * 4; }
    // sum a region on the host in block order (synchronises the stream)
    void host_sum(int region, hipStream_t s, double* out);
    ~Reducer();
};

enum {
    SC_GAMMA = 0,   // z.r of current iteration
    SC_GAMMA_OLD,   // z.r of previous iteration
    SC_ALPHA,       // step length of the last update
    SC_TMP2,
    SC_TMP3,
    SC_DONE,        // flexible CG: 1 once the recursive residual met the tolerance (x is then frozen)
    SC_TOL2,        // flexible CG: (rtol ||b||)^2
    SC_ZERO,        // flexible CG: 1 if b = 0 (the solution is x = 0)
    SC_ITERS,       // flexible CG: iterations that moved x in this solve
    SC_COUNT = 32
};

// ------------------------------------------------------------------ kernel launchers (tt_kernels.hip)
// Elasticity operator on one level.  Coefficient storage CT is double, float or BF16.
enum CoefKind { COEF_F64 = 0, COEF_F32 = 1, COEF_BF16 = 2 };

// Element-local corner numbering of the reference (LinearElasticity.cc:3067-3074)
__host__ __device__ constexpr int corner_id(int x, int y, int z) { return z * 4 + (y == 0 ? (x == 0 ? 0 : 1) : (x == 1 ? 2 : 3)); }
// (i, j, k) of node or element n on an nx x ny x * grid, x fastest: two 32-bit unsigned divisions
// (indices fit in 32 bits; 64-bit division is a long branching sequence on the GPU)
__host__ __device__ inline void grid_ijk(unsigned n, unsigned nx, unsigned ny, int& i, int& j, int& k) {
    const unsigned row = n / nx, kk = row / ny;
    i = (int)(n - row * nx);
    j = (int)(row - kk * ny);
    k = (int)kk;
}
// Element dof order by edges (no kernel uses it; it stays for the test of its invariants): k = 4 t + q (t = 0..5) is dof 3 a + c of corner
// a = sens_corner(q, t >= 3), component c = t mod 3.  Lane group q owns the two x-adjacent corners of one
// element edge (corners 0-1, 3-2, 4-5, 7-6), whose six dofs are consecutive in memory from the edge's
// low-x node.
__host__ __device__ constexpr int sens_corner(int q, int hi) {  // low-x / high-x corner of edge q
    return q == 0 ? hi : q == 1 ? 3 - hi : q == 2 ? 4 + hi : 7 - hi;
}
__host__ __device__ constexpr int sens_dof(int k) {  // k = 4 t + q -> element dof 3 a + c
    return 3 * sens_corner(k & 3, (k >> 2) >= 3) + (k >> 2) % 3;
}
__host__ __device__ constexpr int cx_of(int b) { return (b & 3) == 1 || (b & 3) == 2 ? 1 : 0; }
__host__ __device__ constexpr int cy_of(int b) { return (b & 3) >= 2 ? 1 : 0; }
__host__ __device__ constexpr int cz_of(int b) { return b >> 2; }

struct OpLevel {
    Grid g;
    int coef_kind;         // CoefKind
    const void* kf;        // element stiffness factors (kfac)
    const void* mf;        // element mass factors (mfac)
    const double* KE64;    // 576
    const double* M864;    // 64
    const uint8_t* mask;   // per node clamped bits
    const ModeConst<double>* modes64;  // the element matrices in the symmetry-adapted basis (device)
    const ModeConst<float>* modes32;
    ColSplit split64, split32;  // tile splits of the column kernels, by the precision they compute in
};
// Symmetric coarsest solve on the packed lower triangle (64 x 64 tiles): size of the packed array,
// packing of a full symmetric matrix, and x = A b with per-tile partials (nt (nt + 1) / 2 x 64 each).
long sym_packed_size(int n);
void launch_sym_pack(const double* A, int n, double* P, hipStream_t s);
// Up to order kDenseMvMax the full matrix A is used instead.
constexpr int kDenseMvMax = 1536;
void launch_sym_solve(const double* A, const double* P, const double* b, double* x, int n, double* prow, double* pcol,
                      hipStream_t s);
// Dense N (cK K + cM M) N + I - N of a (coarsest) level from its FP64 element coefficients, on the device
// (row-major n x n, n = g.nd; cleared first).
void launch_dense_coarse(const Grid& g, const double* kf, const double* mf, double cK, double cM, const double* KE,
                         const double* M8, const uint8_t* mask, double* A, hipStream_t s);
// In-place inverse of an m x m (m <= 64) symmetric positive definite block, column-major with leading
// dimension lda (one block, Gauss-Jordan in registers); *info = 1 if a pivot is not positive.
void launch_spd_inv_small(double* A, int m, int lda, int* info, hipStream_t s);
// dst (cols x rows) = src (rows x cols) transposed, column-major with leading dimensions lds, ldd.
void launch_transpose(const double* src, int rows, int cols, int lds, double* dst, int ldd, hipStream_t s);
// y = N.(cK*K + cM*M)(N.u) on free dofs, identity on clamped dofs.  With red: partials of u.y in
// partial region dot_slot (PB_*).  Reductions below likewise take a partial region.
void launch_apply_bc(const OpLevel& L, double cK, double cM, const void* u, void* y, bool fp64, hipStream_t s,
                     Reducer* red = nullptr, int dot_slot = -1);
// r = b - A x
void launch_residual(const OpLevel& L, double cK, double cM, const void* b, const void* x, void* r, bool fp64,
                     hipStream_t s);
// x = c1 D^-1 b and r = b - A x in one pass
void launch_resid_first(const OpLevel& L, double cK, double cM, const void* b, const void* dinv, double c1, void* x,
                        void* r, bool fp64, hipStream_t s);
// r = b - A x (FP64) with the partials of b.b and r.r in two partial regions
void launch_residual_dots(const OpLevel& L, double cK, double cM, const double* b, const double* x, double* r,
                          Reducer& red, int bb_region, int rr_region, hipStream_t s);
// Chebyshev step: r = b - A x; dn = c0*d + c1*dinv.r; xn = x + dn  (d may be null => c0 ignored)
void launch_cheb_step(const OpLevel& L, double cK, double cM, const void* b, const void* x, const void* d,
                      const void* dinv, double c0, double c1, void* xn, void* dn, bool fp64, hipStream_t s);
// split outputs: yk = N.(cK K (N.u)), ym = N.(cM M (N.u))  (FP64)
void launch_apply_split(const OpLevel& L, double cK, double cM, const double* u, double* yk, double* ym,
                        hipStream_t s);
// unmasked K/M apply with arbitrary coefficient arrays (FP64): y = cK*K(kf)u + cM*M(mf)u
void launch_apply_raw(const OpLevel& L, const double* kf, const double* mf, double cK, double cM, const double* u,
                      double* y, hipStream_t s);
// Newmark right-hand side: R = N.( fs*F + sum_i (K-weights, M-weights) applied to u,v,a )
void launch_newmark_rhs(const OpLevel& L, const double* u, const double* v, const double* a, const double* F,
                        double fs, const double wK[3], const double wM[3], double* R, hipStream_t s);
// diagonal of (cK K + cM M) with identity on clamped dofs, inverted
void launch_diag_inv(const OpLevel& L, double cK, double cM, void* dinv, bool fp64, hipStream_t s);

// FCG fused apply: p = z + beta p_old and q = A p = A z + beta q_old, partials of p.q.  Only z is staged with its halo;
// p_old and q_old are read at the owned nodes.  Every block forms beta itself from the z.r and z.q_old partials
// (PB_DOTS): with r = r_prev - alpha q_old, beta = (z.r - z.r_prev) / gamma_old = -alpha z.q_old / gamma_old.
void launch_fcg_apply(const OpLevel& L, double cK, double cM, const double* z, const double* p_old, double* p_new,
                      const double* q_old, double* q_new, Reducer& red, bool first, hipStream_t s);

// vector kernels
void launch_fill(void* x, double v, long n, bool fp64, hipStream_t s);
void launch_copy(const void* src, void* dst, long n, bool src64, bool dst64, hipStream_t s);
void launch_cheb_first(const void* b, const void* dinv, double c1, void* x, long n, bool fp64, hipStream_t s);
// b = (T) r and x = c1 D^-1 b (finest level, r in FP64)
void launch_cheb_first_from64(const double* r, void* b, const void* dinv, double c1, void* x, long n, bool fp64,
                              hipStream_t s);
// first two Chebyshev iterates in one operator apply: x0 = c1_first D^-1 b formed on the fly
// (b = (T) r64 written out when r64 is given), then dn = c0 x0 + c1 D^-1 (b - A x0), xn = x0 + dn
void launch_cheb_first_step(const OpLevel& L, double cK, double cM, const double* r64, void* b, const void* dinv,
                            double c1_first, double c0, double c1, void* xn, void* dn, bool fp64, hipStream_t s);
// last post-smoothing step of the finest level: z (FP64) = x + dn, partials of z.r and z.q_old into PB_DOTS
void launch_cheb_last(const OpLevel& L, double cK, double cM, const void* b, const void* x, const void* d,
                      const void* dinv, double c0, double c1, double* z, const double* r, const double* q, bool first,
                      bool fp64, Reducer& red, hipStream_t s);
// bc = R rf (fine precision fp64; an FP32 fine level may write an FP64 coarse vector, out64)
void launch_restrict(const Grid& fine, const Grid& coarse, const void* rf, const uint8_t* cmask, void* bc,
                     bool fp64, bool out64, hipStream_t s);
// xf += sum_l P_l xc[l]: the corrections of the n coarser levels coarse[0..n-1] (each 2:1 from the one before, the first
// from `fine`), in the fine precision except that an FP32 fine level may read an FP64 last one (last64)
void launch_prolong_chain(const Grid& fine, int n, const Grid* const* coarse, const void* const* xc,
                          const uint8_t* fmask, void* xf, bool fp64, bool last64, hipStream_t s);
void launch_coarsen_coef(const Grid& fine, const Grid& coarse, const double* kf_f, const double* mf_f, double* kf_c,
                         double* mf_c, hipStream_t s);
void launch_convert_coef(const double* src, void* dst, long n, int kind, hipStream_t s);
void launch_interp(const double* x, long n, int sInt, double Emin, double Emax, double pK, int mInt, double Rmin,
                   double Rmax, double pM, const double* P, double* kf, double* mf, double* dkf, double* dmf,
                   double* Pkf, double* Pmf, hipStream_t s);

// dots (FP64): results land in red.scal[slot..]
void launch_dot(const double* a, const double* b, long n, Reducer& red, int slot, hipStream_t s);
// Q_k.a, Q_k.b, Q_k.c for the nq <= 8 vectors Q_k = Q + k*n, k0 <= k < k0 + nq, in one pass over a, b, c:
// block partials into part[(k*1024 + block)*3 + i]; returns the number of blocks (at most 1024)
int launch_proj3(const double* Q, int k0, int nq, const double* a, const double* b, const double* c, long n,
                 double* part, hipStream_t s);
// Modified Gram-Schmidt of w against the k orthonormal vectors V_i = V + i*n, then w /= ||w||, on the device: h[0..k-1]
// receive the coefficients and h[k] = ||w|| (w stays as it is if that is 0).  Groups of kMgsGroup vectors share a
// pass over w; G (kMgsMax x kMgsMax, device, kept between calls while V grows) holds the dots of vectors of one
// group, from which the group's coefficients follow one after the other.  part: 2 x kMgsBlocks x (kMgsGroup + 1).
constexpr int kMgsGroup = 8, kMgsBlocks = 256, kMgsMax = 32;
void launch_mgs(double* w, const double* V, int k, long n, double* G, double* h, double* part, hipStream_t s);
// out[o] = sum_k c[o][k] Q_k for nout <= 3 outputs and nb <= 64 vectors Q_k = Q + k*n, one pass over Q
struct Expand3 {
    const double* Q;
    double* out[3];
    double c[3][64];
    int nb, nout;
};
void launch_expand3(const Expand3& e, long n, hipStream_t s);
// out[0] += sum_k c[0][k] Q_k
void launch_axpy_multi(const Expand3& e, long n, hipStream_t s);
// partials of z.r and z.q_old (PB_DOTS)
void launch_fcg_dots(const double* z, const double* r, const double* q_old, long n, Reducer& red, bool first,
                     hipStream_t s);
// Flexible-CG (re)start from the b.b and r.r partial regions: device tolerance (rtol ||b||)^2, the
// b = 0 flag, and whether the current x already meets the tolerance.
// reset_iters: a new solve (SC_ITERS = 0) rather than a restart of the same one.
void launch_fcg_init(Reducer& red, int bb_region, int rr_region, double rtol2, bool reset_iters, hipStream_t s);
// x += alpha p, r -= alpha q with alpha = gamma / p.q, unless x already met the tolerance (set at the
// (re)start, or by the previous update's r.r after its first iteration): then alpha = 0 from there on,
// so the result does not depend on when the host looks at the residual.  x = 0 if b = 0.  Every block forms alpha
// itself from the p.q partials and the previous update's r.r; odd: the parity of the iteration (its r.r partials go to
// region rr_region(odd), the previous update's are in the other one).
inline int rr_region(bool odd) { return odd ? PB_RR2 : PB_RR; }
// With dinv, the partials of z.r and z.q for the next direction (z = D^-1 r of the new r) go to PB_DOTS: the Jacobi
// preconditioner needs no kernel of its own.
void launch_fcg_update(double* x, const double* p, double* r, const double* q, long n, Reducer& red, bool first,
                       bool odd, hipStream_t s, const double* dinv = nullptr);
void launch_jacobi(const double* dinv, const double* r, double* z, long n, hipStream_t s);
// power iteration: x = dinv.Ax with partials of ||x||^2 in PB_MISC; then x /= ||x||
void launch_norm_power(const void* Ax, const void* dinv, void* x, long n, Reducer& red, bool fp64, hipStream_t s);
void launch_scale_by_norm(void* x, long n, Reducer& red, bool fp64, hipStream_t s);

// Newmark corrector: vn = a0 v + a1 a + a2 (un - u); an = -a3 v - a4 a + a5 (un - u).  With nh > 0 it
// also writes the nh vectors hout[0] = a, hout[j] = hin[j - 1] (each n long, stored n apart).
struct Extrap;
// With next (its coefficients; its vectors are ignored) and gout, the kernel also writes the next step's
// initial guess sum_k c_k w_k over w = (un, vn, an, a, hin[0], hin[1]) (the new state's u, v, a and history),
// in k_extrapolate's order of operations.
void launch_newmark_update(const double* u, const double* v, const double* a, const double* un, double* vn,
                           double* an, const double* c, long n, const double* hin, double* hout, int nh,
                           hipStream_t s, const Extrap* next = nullptr, double* gout = nullptr);
// adjoint combination (see transient.cpp)
void launch_adjoint_combine(const double* Kl, const double* Ml, const double* hdu, const double* hddu,
                            const double* hdddu, const double* mun, const double* nun, const uint8_t* mask,
                            const double* coef, bool terminal, double* mu, double* nu, double* rhs, long nn,
                            hipStream_t s);
void launch_adjoint0_rhs(const double* Kl, const double* Ml, const double* hdddu, const double* mun,
                         const double* nun, const uint8_t* mask, const double* coef, double* rhs, long nn,
                         hipStream_t s);
// objective gradient wrt state for objectives 0..2 (diagonal with region counts)
void launch_hdiag(const double* w, const double* cnt, double dt, double* h, long nn, hipStream_t s);
void launch_region_count(const Grid& g, const double* P, double* cnt, hipStream_t s);

// sensitivities and objective (per time step); accumulates into df, objective partials per block
struct SensArgs {
    Grid g;
    const ModeConst<double>* modes;
    const double *kf, *mf, *dkf, *dmf, *P;
    const double *lam, *u, *v, *a, *ub, *vb, *ab;
    double wK[4];  // coefficients of (u, ub, vb, ab) in w_K
    double wM[4];  // coefficients of (u, ub, vb, ab) in w_M
    double dt, dalpha, dbeta;
    int objective;
    int mode;      // 0: general step (lambda), 1: t = 0 step (nu0 with dK u0 + dC v0 + dM a0)
    double* df;
};
long sens_blocks(const Grid& g);  // objective partials written to fx_out
void launch_sens(const SensArgs& a, double* fx_out, hipStream_t s);

// PDE filter (scalar Helmholtz on nodes)
// The filter's operator R^2 (Kx My Mz + Mx Ky Mz + Mx My Kz) + Mx My Mz by its 1-D factors.
struct FilterOp {
    double h[3], R2;
};
// r = rhs - A U, partials of r.r (PB_MISC2), of z.r with z = D^-1 r (PB_DOTS) and, with bb, of rhs.rhs (PB_MISC)
long filter_blocks(const Grid& g);  // partials written by the two launches below
void launch_filter_residual(const Grid& g, const FilterOp& f, const double* U, const double* rhs, const double* dinv,
                            double* r, Reducer& red, bool bb, hipStream_t s);
// Jacobi-preconditioned CG direction and product: p = z + beta p_old with z = D^-1 r, q = A p, partials of p.q
void launch_filter_direction(const Grid& g, const FilterOp& f, const double* r, const double* dinv, const double* p_old,
                             double* p_new, double* q, Reducer& red, bool first, hipStream_t s);
void launch_filter_T(const Grid& g, const double* x, double scale, double* rhs, hipStream_t s);
void launch_filter_Tt(const Grid& g, const double* U, double* out, hipStream_t s);
void launch_filter_diag(const Grid& g, const double* kf, double* dinv, hipStream_t s);
void launch_clamp_project(const double* xt_in, double* xt, double* xp, long n, int projection, double beta,
                          double eta, hipStream_t s);
void launch_project_chain(const double* xt, double* df, double* dg, long n, double beta, double eta,
                          hipStream_t s);
// reductions over element arrays
void launch_sum(const double* x, long n, Reducer& red, int slot, hipStream_t s);
// the same block partial sums of x written to `partials` (room for `capacity` values; at most 256 are
// needed, whatever n is); returns the number of blocks
int launch_sum_partials(const double* x, long n, double* partials, int capacity, hipStream_t s);
void launch_mnd(const double* x, long n, Reducer& red, int slot, hipStream_t s);

// MMA kernels (m = 1)
struct MMADev {
    long n;
    double *L, *U, *alpha, *beta, *p0, *q0, *pij, *qij, *xo1, *xo2;
};
void launch_mma_gensub(const MMADev& m, const double* x, const double* df, const double* dg, const double* xmin,
                       const double* xmax, int k, double asyminit, double asymdec, double asyminc, Reducer& red,
                       hipStream_t s);
void launch_mma_xyz_grad_hess(const MMADev& m, double lam, double* x, Reducer& red, hipStream_t s);
void launch_mma_xyz_res(const MMADev& m, double lam, double* x, Reducer& red, hipStream_t s);
void launch_mma_movelimit(const double* x, double* xmin, double* xmax, long n, double Xmin, double Xmax,
                          double movlim, hipStream_t s);
void launch_mma_change(const double* x, double* xold, long n, Reducer& red, int slot, hipStream_t s);
void launch_mma_kkt(const double* x, const double* df, const double* dg, const double* xmin, const double* xmax,
                    long n, double lam, Reducer& red, hipStream_t s);
// x_i in [-1, 1) from a counter-based hash of (seed, i): deterministic, generated on the device
void launch_fill_hash(void* x, long n, unsigned long long seed, bool fp64, hipStream_t s);
// x = N.x (clamped dofs of the node mask set to 0)
void launch_mask_dofs(double* x, const uint8_t* mask, long nd, hipStream_t s);
void launch_scale(double* x, long n, double a, hipStream_t s);
// out = a*x + b*y (out may alias x or y)
void launch_lincomb(double a, const double* x, double b, const double* y, double* out, long n, hipStream_t s);
// out = sum_k c[k] v[k] over the m <= 8 vectors of e (polynomial extrapolation of a sequence)
struct Extrap {
    const double* v[8];
    double c[8];
    int m;
};
void launch_extrapolate(const Extrap& e, double* out, long n, hipStream_t s);

}  // namespace tt
