// Element matrices of the trilinear hex8 on an axis-aligned box element.
//
// Same integrals as the reference's Hex8IsoparametricKE/ME (LinearElasticity.cc:
// 3089-3333) and closed-form PDE-filter matrix (PDEFilter.cc:485-578): 2x2x2
// Gauss quadrature of B^T C B (E = 1), of N^T N (density 1), and of
// R^2 grad N . grad N + N N.  For a box element the Jacobian is diagonal,
// so shape-function gradients are the parametric ones scaled by 2/h.
#include <cmath>
#include <cstring>

#include "tt_internal.h"

namespace tt {

// Gauss abscissa as written in the reference (LinearElasticity.cc:3150)
static const double kGP = 0.577350269189626;

static const int kSx[8] = {-1, 1, 1, -1, -1, 1, 1, -1};
static const int kSy[8] = {-1, -1, 1, 1, -1, -1, 1, 1};
static const int kSz[8] = {-1, -1, -1, -1, 1, 1, 1, 1};

struct GaussPoint {
    double N[8], dx[8], dy[8], dz[8], w;
};

static GaussPoint gauss_point(double xi, double eta, double zeta, double hx, double hy, double hz) {
    GaussPoint g;
    for (int a = 0; a < 8; a++) {
        const double fx = 1.0 + kSx[a] * xi, fy = 1.0 + kSy[a] * eta, fz = 1.0 + kSz[a] * zeta;
        g.N[a] = 0.125 * fx * fy * fz;
        g.dx[a] = 0.125 * kSx[a] * fy * fz * (2.0 / hx);
        g.dy[a] = 0.125 * kSy[a] * fx * fz * (2.0 / hy);
        g.dz[a] = 0.125 * kSz[a] * fx * fy * (2.0 / hz);
    }
    g.w = 0.125 * hx * hy * hz;  // unit weights times det J
    return g;
}

void hex8_stiffness(double hx, double hy, double hz, double nu, double* ke) {
    const double lam = nu / ((1.0 + nu) * (1.0 - 2.0 * nu));
    const double mu = 1.0 / (2.0 * (1.0 + nu));
    double D[6][6] = {};
    for (int i = 0; i < 3; i++) {
        for (int j = 0; j < 3; j++) D[i][j] = lam;
        D[i][i] = lam + 2.0 * mu;
        D[3 + i][3 + i] = mu;
    }
    std::memset(ke, 0, sizeof(double) * 576);
    const double gp[2] = {-kGP, kGP};
    for (int iz = 0; iz < 2; iz++)
        for (int iy = 0; iy < 2; iy++)
            for (int ix = 0; ix < 2; ix++) {
                GaussPoint g = gauss_point(gp[ix], gp[iy], gp[iz], hx, hy, hz);
                // strain rows: xx, yy, zz, xy, yz, zx
                double B[6][24] = {};
                for (int a = 0; a < 8; a++) {
                    const int u = 3 * a, v = 3 * a + 1, w = 3 * a + 2;
                    B[0][u] = g.dx[a];
                    B[1][v] = g.dy[a];
                    B[2][w] = g.dz[a];
                    B[3][u] = g.dy[a];
                    B[3][v] = g.dx[a];
                    B[4][v] = g.dz[a];
                    B[4][w] = g.dy[a];
                    B[5][u] = g.dz[a];
                    B[5][w] = g.dx[a];
                }
                double DB[6][24];
                for (int r = 0; r < 6; r++)
                    for (int c = 0; c < 24; c++) {
                        double s = 0.0;
                        for (int k = 0; k < 6; k++) s += D[r][k] * B[k][c];
                        DB[r][c] = s;
                    }
                for (int i = 0; i < 24; i++)
                    for (int j = 0; j < 24; j++) {
                        double s = 0.0;
                        for (int k = 0; k < 6; k++) s += B[k][i] * DB[k][j];
                        ke[24 * i + j] += g.w * s;
                    }
            }
}

void hex8_mass(double hx, double hy, double hz, double* m8) {
    std::memset(m8, 0, sizeof(double) * 64);
    const double gp[2] = {-kGP, kGP};
    for (int iz = 0; iz < 2; iz++)
        for (int iy = 0; iy < 2; iy++)
            for (int ix = 0; ix < 2; ix++) {
                GaussPoint g = gauss_point(gp[ix], gp[iy], gp[iz], hx, hy, hz);
                for (int a = 0; a < 8; a++)
                    for (int b = 0; b < 8; b++) m8[8 * a + b] += g.w * g.N[a] * g.N[b];
            }
}

// K~ = H K H' / 64 and M~ = H M H' / 64 with the 8 x 8 sign matrix H (per component), so that K = H' K~ H.  Mode
// m = a + 2 b + 4 c has sign (2 i - 1) along each direction whose bit is set.  Box elements are symmetric under
// the three reflections: K~ has no entries besides the blocks kept here, and M~ is diagonal, with a third per
// odd direction.  (Summed in extended precision: the constants carry the matrices' rounding only.)
void hex8_modes(const double* ke, const double* m8, ModeConst<double>& mc) {
    double H[8][8];
    for (int m = 0; m < 8; m++)
        for (int a = 0; a < 8; a++)
            H[m][a] = ((m & 1) ? kSx[a] : 1) * ((m & 2) ? kSy[a] : 1) * ((m & 4) ? kSz[a] : 1);
    auto K = [&](int ci, int mi, int cj, int mj) {
        long double s = 0.0L;
        for (int a = 0; a < 8; a++)
            for (int b = 0; b < 8; b++) s += (long double)(H[mi][a] * H[mj][b]) * ke[(3 * a + ci) * 24 + 3 * b + cj];
        return (double)(s / 64.0L);
    };
    struct CM {
        int c, m;
    };
    auto block = [&](const CM* x, int n, double* out) {
        for (int i = 0; i < n; i++)
            for (int j = i; j < n; j++) *out++ = K(x[i].c, x[i].m, x[j].c, x[j].m);
    };
    const CM nn[3] = {{0, 1}, {1, 2}, {2, 4}}, tt[3] = {{0, 6}, {1, 5}, {2, 3}};
    const CM qq[3][2] = {{{1, 3}, {2, 5}}, {{0, 3}, {2, 6}}, {{0, 5}, {1, 6}}};
    const CM ss[3][2] = {{{0, 2}, {1, 1}}, {{0, 4}, {2, 1}}, {{1, 4}, {2, 2}}};
    block(nn, 3, mc.n);
    block(tt, 3, mc.t);
    for (int k = 0; k < 3; k++) {
        block(qq[k], 2, mc.q[k]);
        block(ss[k], 2, mc.s[k]);
        mc.d[k] = K(k, 7, k, 7);
    }
    const int of[4] = {0, 1, 3, 7};  // one mode of each number of odd directions
    for (int k = 0; k < 4; k++) {
        long double s = 0.0L;
        for (int a = 0; a < 8; a++)
            for (int b = 0; b < 8; b++) s += (long double)(H[of[k]][a] * H[of[k]][b]) * m8[8 * a + b];
        mc.m[k] = (double)(s / 64.0L);
    }
}

void upload_modes(const double* ke, const double* m8, DBuf<ModeConst<double>>& d64, DBuf<ModeConst<float>>& d32) {
    ModeConst<double> mc;
    hex8_modes(ke, m8, mc);
    ModeConst<float> mf;
    static_assert(sizeof(mc) == 37 * sizeof(double) && sizeof(mf) == 37 * sizeof(float), "37 constants");
    for (int i = 0; i < 37; i++) reinterpret_cast<float*>(&mf)[i] = (float)reinterpret_cast<const double*>(&mc)[i];
    d64.alloc(1);
    d32.alloc(1);
    TT_HIP(hipMemcpy(d64.p, &mc, sizeof(mc), hipMemcpyHostToDevice));
    TT_HIP(hipMemcpy(d32.p, &mf, sizeof(mf), hipMemcpyHostToDevice));
}

void hex8_helmholtz(double hx, double hy, double hz, double R, double* kf) {
    std::memset(kf, 0, sizeof(double) * 64);
    const double q = 1.0 / std::sqrt(3.0);
    const double gp[2] = {-q, q};
    for (int iz = 0; iz < 2; iz++)
        for (int iy = 0; iy < 2; iy++)
            for (int ix = 0; ix < 2; ix++) {
                GaussPoint g = gauss_point(gp[ix], gp[iy], gp[iz], hx, hy, hz);
                for (int a = 0; a < 8; a++)
                    for (int b = 0; b < 8; b++)
                        kf[8 * a + b] += g.w * (R * R * (g.dx[a] * g.dx[b] + g.dy[a] * g.dy[b] + g.dz[a] * g.dz[b]) +
                                                g.N[a] * g.N[b]);
            }
}

}  // namespace tt
