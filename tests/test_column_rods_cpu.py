"""Host side of the operator's tile splits (csrc/tt_colplan.cpp) on rods, grids of few columns and many planes, checked on
the CPU by small programs.

* col_bc_flags takes time in proportion to the grid: a rod of 400,001 planes in 200,000 parts is done at once (formed
  part by part for every plane it takes minutes), with the flags of a direct test of every part's planes.
* make_col_plan cuts a block's planes into strands where the cross-section's columns fit the block twice or more, as many
  as its 256 threads and 1,024 staging slots hold, and into one otherwise.
"""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "topopt_in_petsc_transient_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"

FLAGS = r"""
#include "tt_colplan.cpp"
#include <cstdio>
using namespace tt;
static int flags(const Grid& g, const ColPlan& p, int every) {  // every `every`-th plane has a clamped node
    std::vector<uint8_t> m(g.nn, 0), f;
    for (int k = 0; k < g.nz; k += every) m[(size_t)g.nx * g.ny * k + k % (g.nx * g.ny)] = 1;
    col_bc_flags(g, p, m, f);
    int bad = (int)f.size() != p.ntiles();
    for (int c = 0; c < p.tz; c++) {
        const int k0 = (int)((long)c * g.nz / p.tz), k1 = (int)((long)(c + 1) * g.nz / p.tz);
        int any = 0;
        for (int k = std::max(k0 - 1, 0); k <= std::min(k1, g.nz - 1); k++) any |= k % every == 0;
        bad += any != f[c];
    }
    return bad;
}
int main() {
    int bad = 0;
    const Grid g = make_grid(1, 1, 400000, 1, 1, 1);
    const ColPlan p{3, 2, 2, 1, 1, 200000}, q{3, 2, 2, 1, 1, 7};
    bad += flags(g, p, 1000) + flags(g, p, 3) + flags(g, q, 1000) + flags(g, q, 399999);
    const Grid h = make_grid(3, 2, 40, 1, 1, 1);
    for (int tz = 1; tz <= h.nz; tz++) bad += flags(h, ColPlan{5, 4, 3, 1, 1, tz}, 11);
    printf("bad %d\n", bad);
    return bad != 0;
}
"""

STRANDS = r"""
#include "tt_colplan.cpp"
#include <cstdio>
using namespace tt;
int main() {
    int bad = 0;
    const int cs[][2] = {{1, 1}, {2, 2}, {3, 3}, {5, 5}, {7, 7}, {8, 8}, {9, 9}, {1, 7}, {7, 1}, {2, 20}, {20, 2}, {1, 39}, {3, 24},
                         {10, 10}, {40, 20}, {128, 64}};
    for (auto& c : cs)
        for (long n : {45000, 70000, 900000})
            for (int d = 0; d < 2; d++) {
                const Grid g = make_grid(c[0], c[1], (int)(n / ((c[0] + 1) * (c[1] + 1))), 1, 1, 1);
                const ColPlan p = make_col_plan(g, d != 0);
                const int cols = p.cx * (p.by + 1), dofs = 3 * (p.bx + 2) * (p.by + 2);
                int e = p.strands < 1 || p.strands * cols > 256 || p.strands * dofs > 1024 ||
                        (p.strands > 1 && (p.tx * p.ty != 1 || p.bx != g.nx || p.by != g.ny));
                // a tile of the whole cross-section is filled up; of a small one (half the threads idle) it is taken
                if (p.tx * p.ty == 1) e += (p.strands + 1) * cols <= 256 && (p.strands + 1) * dofs <= 1024;
                if (2 * (g.nx + 1) * (g.ny + 1) <= 170 && 6 * (g.nx + 2) * (g.ny + 2) <= 1024) e += p.strands < 2;
                if (e) printf("%d x %d, %ld, %d: strands %d, %d columns, %d dofs\n", c[0], c[1], n, d, p.strands, cols, dofs);
                bad += e;
            }
    printf("bad %d\n", bad);
    return bad != 0;
}
"""


def _run(tmp_path, name, prog, timeout):
    src = tmp_path / (name + ".cpp")
    src.write_text(prog)
    exe = tmp_path / name
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-xhip", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=timeout)
    assert r.returncode == 0 and "bad 0" in r.stdout, r.stdout


def test_flags_of_a_rod(tmp_path):
    _run(tmp_path, "flags", FLAGS, 20)


def test_strands_of_a_rod(tmp_path):
    _run(tmp_path, "strands", STRANDS, 60)
