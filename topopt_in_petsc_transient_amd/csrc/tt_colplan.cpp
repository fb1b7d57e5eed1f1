// Tile splits of the column kernels (tt_apply_cols.inc).  Host code, run once per grid.
#include <algorithm>
#include <cmath>

#include "tt_internal.h"

namespace tt {

// Tile split of one grid.  A block's planes pass one after the other, so its time is (planes + 2) times the time of a
// plane: a latency that grows slowly with the blocks sharing a CU, plus the cache lines the tile's rows touch (a narrow
// tile reads more halo).  The constants are fitted to 170 splits on each of 8 grids between 97x51x43 and 320x160x160
// elements (FP64 to the plain and the flexible-CG apply alike; rms error 6 and 9 %).  The columns of a tile (cx x cy <=
// 256 threads, one halo row and column) and the planes per block trade halo work against blocks in flight: the split
// with the least modelled time is taken.  Against a model with a plane bound by issue alone (FP64 apply, FP32 apply,
// flexible-CG apply; us): 192x96x96 40.6 -> 39.4, 26.7 -> 22.6, 62 -> 57; 320x160x160 171 -> 163, 95 -> 78, 305 -> 283;
// 40x40x300 17.7 -> 17.1, 12.3 -> 11.3, 23.4 -> 22.2; 128x64x64 and smaller as they were.
// Grids of up to kBoxNodes nodes take the one-shot kernel: at 1,377 nodes (16x8x8) an FP64 apply takes 3.5 us there against
// 5.6 us in columns, at 30,625 (48x24x24) 4.5 against 5.8 (flexible-CG apply 6.8 against 8.5, FP32 3.8 against 5.0); at
// 70,785 (64x32x32) 6.9 against 7.1, and the flexible-CG apply 13.4 against 10.1.  (Longer rods march in strands: at 60,016
// nodes, 3x3x3750, one shot takes 4.8 us, flexible-CG apply 7.6, and strands 7.5 and 11.1; at 300,004, 1x1x75000, 50 and 226
// against 19 and 26, every block summing all blocks' partials.)
constexpr long kBoxNodes = 40000;
ColPlan make_col_plan(const Grid& g, bool fp64) {
    constexpr double cus = 256.0;
    const int resident = fp64 ? 2 : 3;  // blocks per CU (2 in the first Chebyshev step from FP64, FP32's largest form)
    // us per plane with r blocks on the CU, and per r and 100 lines of 128 bytes touched
    const double base[3] = {fp64 ? 1.4 : 0.83, fp64 ? 1.95 : 1.03, 1.25}, lines = fp64 ? 0.17 : 0.013;
    const double tail = fp64 ? 0.3 : 0.35;  // of a full CU's plane: blocks of the last round left alone
    if (g.nn <= kBoxNodes) return ColPlan{0, 4, 4, (g.nx + 3) / 4, (g.ny + 3) / 4, (g.nz + 3) / 4};
    ColPlan best{};
    double cost = 1e300;
    for (int cx = std::min(3, g.nx + 1); cx <= std::min(34, g.nx + 1); cx++) {
        const int bx = cx - 1, tx = (g.nx + bx - 1) / bx;
        const int cymax = std::min({256 / cx, 1024 / (3 * (cx + 1)) - 1, g.ny + 1});
        for (int cy = std::min(3, cymax); cy <= cymax; cy++) {
            const int by = cy - 1, ty = (g.ny + by - 1) / by;
            const double row = (std::min(cx, g.nx) + 1) * 3.0 * (fp64 ? 8 : 4) / 128.0 + 1.0;
            // a tile of the whole cross-section with room for more beside it: its planes in strands (ROD in tt_apply_cols.inc)
            const int strands = tx * ty == 1 ? std::max(1, std::min(256 / (cx * cy), 1024 / (3 * (cx + 1) * (cy + 1)))) : 1;
            const double touched = lines * strands * row * (std::min(cy, g.ny) + 1) / 100.0;
            auto plane = [&](int r) { return base[r - 1] + r * touched; };
            for (int nk = 1;;) {  // planes per block: the fewest that give each number of blocks in z
                const int tz = (g.nz + nk - 1) / nk;
                const double nt = (double)tx * ty * tz, per = nt / cus;
                const int r = (int)std::ceil(per);
                // (between splits of one modelled time, the one with fewer blocks)
                const double c = 1e-4 * nt + ((strands == 1 ? nk : (nk + strands - 1) / strands) + 2) * (r <= resident ? plane(r) : plane(resident) * (tail + per / resident));
                if (c < cost) {
                    cost = c;
                    best = ColPlan{cx, bx, by, tx, ty, tz, strands};
                }
                if (tz == 1) break;
                nk = (g.nz + tz - 2) / (tz - 1);
            }
        }
    }
    return best;
}

void col_bc_flags(const Grid& g, const ColPlan& p, const std::vector<uint8_t>& mask, std::vector<uint8_t>& f) {
    f.assign(p.ntiles(), 0);
    // tile a (b nodes per tile) stages nodes a b - 1 .. (a + 1) b
    auto range = [](int i, int b, int nt, int& lo, int& hi) {
        lo = std::max(0, (i + b - 1) / b - 1);
        hi = std::min(nt - 1, (i + 1) / b);
    };
    // the parts that stage node plane k: zlo[k] .. zhi[k] (one pass over the parts, which follow one another: a rod's
    // grid has thousands of both)
    std::vector<int> zlo(g.nz, p.tz), zhi(g.nz, -1);
    for (int c = 0; c < p.tz; c++) {
        const int k0 = (int)((long)c * g.nz / p.tz), k1 = (int)((long)(c + 1) * g.nz / p.tz);
        for (int k = std::max(k0 - 1, 0); k <= std::min(k1, g.nz - 1); k++) {
            zlo[k] = std::min(zlo[k], c);
            zhi[k] = c;
        }
    }
    for (int k = 0; k < g.nz; k++)
        for (int j = 0; j < g.ny; j++)
            for (int i = 0; i < g.nx; i++) {
                if (!mask[i + (size_t)g.nx * (j + (size_t)g.ny * k)]) continue;
                int a0, a1, b0, b1;
                range(i, p.bx, p.tx, a0, a1);
                range(j, p.by, p.ty, b0, b1);
                for (int c = zlo[k]; c <= zhi[k]; c++)
                    for (int b = b0; b <= b1; b++)
                        for (int a = a0; a <= a1; a++) f[a + (size_t)p.tx * (b + (size_t)p.ty * c)] = 1;
            }
}

void ColSplitStore::build(const Grid& g, const std::vector<uint8_t>& mask) {
    for (int d = 0; d < 2; d++) {
        ColSplit& s = d ? s64 : s32;
        s.plan = make_col_plan(g, d != 0);
        if (s.plan.cx == 0) continue;  // (the one-shot kernel reads the mask itself)
        std::vector<uint8_t> f;
        col_bc_flags(g, s.plan, mask, f);
        flags[d].alloc(f.size());
        TT_HIP(hipMemcpy(flags[d].p, f.data(), f.size(), hipMemcpyHostToDevice));
        s.bc = flags[d].p;
    }
}

}  // namespace tt
