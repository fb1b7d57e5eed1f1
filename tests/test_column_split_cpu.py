"""Host side of the column kernels (csrc/tt_colplan.cpp, csrc/tt_element.cpp), checked on the CPU by a small program.

* make_col_plan: a tile's columns fit the block's 256 threads and its staged plane the 1024 staging slots, the tiles
  cover the grid without an empty one, for grids from one element up and both precisions.
* col_bc_flags: equal to a direct test of every tile's node box, for the two boundary masks.
* hex8_modes: K = H' K~ H and M = H' M~ H with the kept blocks alone give the element matrices back, to rounding.
"""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "topopt_in_petsc_transient_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"

PROG = r"""
#include "tt_colplan.cpp"
#include "tt_element.cpp"
#include <cstdio>
using namespace tt;
static int modes(double hx, double hy, double hz, double nu) {
    double ke[576], m8[64];
    hex8_stiffness(hx, hy, hz, nu, ke);
    hex8_mass(hx, hy, hz, m8);
    ModeConst<double> c;
    hex8_modes(ke, m8, c);
    static double Kt[24][24], H[8][8];
    for (auto& r : Kt) for (double& v : r) v = 0.0;
    for (int m = 0; m < 8; m++)
        for (int a = 0; a < 8; a++) {
            const int p[3] = {cx_of(a), cy_of(a), cz_of(a)};
            H[m][a] = 1.0;
            for (int d = 0; d < 3; d++) if (m >> d & 1) H[m][a] *= 2 * p[d] - 1;
        }
    auto put = [&](const int* id, int n, const double* v) {  // id = 3 mode + component
        for (int i = 0; i < n; i++)
            for (int j = i; j < n; j++, v++) Kt[id[i]][id[j]] = Kt[id[j]][id[i]] = *v;
    };
    auto id = [](int comp, int x, int y, int z) { return 3 * (x + 2 * y + 4 * z) + comp; };
    const int n[3] = {id(0,1,0,0), id(1,0,1,0), id(2,0,0,1)}, t[3] = {id(0,0,1,1), id(1,1,0,1), id(2,1,1,0)};
    const int q[3][2] = {{id(1,1,1,0), id(2,1,0,1)}, {id(0,1,1,0), id(2,0,1,1)}, {id(0,1,0,1), id(1,0,1,1)}};
    const int s[3][2] = {{id(0,0,1,0), id(1,1,0,0)}, {id(0,0,0,1), id(2,1,0,0)}, {id(1,0,0,1), id(2,0,1,0)}};
    put(n, 3, c.n);
    put(t, 3, c.t);
    for (int k = 0; k < 3; k++) {
        put(q[k], 2, c.q[k]);
        put(s[k], 2, c.s[k]);
        Kt[21 + k][21 + k] = c.d[k];
    }
    double ek = 0, em = 0, mk = 0, mm = 0;
    for (int a = 0; a < 8; a++)
        for (int b = 0; b < 8; b++) {
            double m = 0;
            for (int w = 0; w < 8; w++) m += H[w][a] * H[w][b] * c.m[(w & 1) + (w >> 1 & 1) + (w >> 2)];
            em = std::max(em, std::fabs(m - m8[8 * a + b]));
            mm = std::max(mm, std::fabs(m8[8 * a + b]));
            for (int i = 0; i < 3; i++)
                for (int j = 0; j < 3; j++) {
                    double k = 0;
                    for (int w = 0; w < 8; w++)
                        for (int v = 0; v < 8; v++) k += H[w][a] * Kt[3 * w + i][3 * v + j] * H[v][b];
                    const double ref = ke[(3 * a + i) * 24 + 3 * b + j];
                    ek = std::max(ek, std::fabs(k - ref));
                    mk = std::max(mk, std::fabs(ref));
                }
        }
    if (ek > 5e-15 * mk || em > 5e-15 * mm) { printf("modes %g %g %g nu %g: %g %g\n", hx, hy, hz, nu, ek / mk, em / mm); return 1; }
    return 0;
}
static int plan(int ex, int ey, int ez) {
    const Grid g = make_grid(ex, ey, ez, 1, 1, 1);
    int bad = 0;
    for (int d = 0; d < 2; d++) {
        const ColPlan p = make_col_plan(g, d != 0);
        if (p.cx == 0) {  // the one-shot kernel's 4 x 4 x 4 tiles
            bad += p.tx != (ex + 4) / 4 || p.ty != (ey + 4) / 4 || p.tz != (ez + 4) / 4 || g.nn > kBoxNodes;
            continue;
        }
        const int cy = p.by + 1;
        bad += g.nn <= kBoxNodes;
        bad += p.bx < 1 || p.by < 1 || p.cx != p.bx + 1 || p.cx * cy > 256 || 3 * (p.cx + 1) * (cy + 1) > 1024;
        bad += p.tx * p.bx < g.nx || (p.tx - 1) * p.bx >= g.nx || p.ty * p.by < g.ny || (p.ty - 1) * p.by >= g.ny;
        bad += p.tz < 1 || p.tz > g.nz;
        for (int b = 0; b < 2; b++) {
            std::vector<uint8_t> m(g.nn, 0), f;
            for (int k = 0; k < g.nz; k++)
                for (int j = 0; j < g.ny; j++)
                    for (int i = 0; i < g.nx; i++)
                        m[i + (size_t)g.nx * (j + (size_t)g.ny * k)] =
                            b ? (i == 0 ? 7 : 0) : ((i == 0 ? 3 : 0) | (i == g.nx - 1 && k == 0 ? 6 : 0));
            col_bc_flags(g, p, m, f);
            for (int t = 0; t < p.ntiles(); t++) {
                const int a = t % p.tx, c = t / p.tx % p.ty, z = t / (p.tx * p.ty);
                const int k0 = (int)((long)z * g.nz / p.tz), k1 = (int)((long)(z + 1) * g.nz / p.tz);
                bad += k1 <= k0;
                int any = 0;
                for (int k = std::max(k0 - 1, 0); k <= std::min(k1, g.nz - 1); k++)
                    for (int j = std::max(c * p.by - 1, 0); j <= std::min((c + 1) * p.by, g.ny - 1); j++)
                        for (int i = std::max(a * p.bx - 1, 0); i <= std::min((a + 1) * p.bx, g.nx - 1); i++)
                            any |= m[i + (size_t)g.nx * (j + (size_t)g.ny * k)];
                bad += (any != 0) != (f[t] != 0);
            }
        }
    }
    if (bad) printf("grid %d %d %d: %d\n", ex, ey, ez, bad);
    return bad;
}
int main() {
    int bad = 0;
    const int ext[] = {1, 2, 3, 7, 8, 15, 16, 17, 31, 64, 97};
    for (int x : ext) for (int y : ext) for (int z : ext) if (x * y * z <= 150000) bad += plan(x, y, z);
    bad += plan(128, 64, 64) + plan(30000, 1, 1) + plan(1, 11000, 2) + plan(2, 1, 9000) + plan(300, 11, 12);
    bad += modes(0.1, 0.1, 0.1, 0.3) + modes(1, 1, 1, 0.0) + modes(0.01, 0.2, 3.0, 0.45) + modes(2, 0.3, 0.3, -0.4);
    printf("bad %d\n", bad);
    return bad != 0;
}
"""


def test_column_split_and_modes(tmp_path):
    src = tmp_path / "colsplit.cpp"
    src.write_text(PROG)
    exe = tmp_path / "colsplit"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-xhip", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and "bad 0" in r.stdout, r.stdout
