"""Host side of the operator's tile splits (csrc/tt_colplan.cpp) on rods, grids of few columns and many planes, checked on
the CPU by small programs.

* col_bc_flags takes time in proportion to the grid: a rod of 400,001 planes in 200,000 parts is done at once (formed
  part by part for every plane it takes minutes), with the flags of a direct test of every part's planes.
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
