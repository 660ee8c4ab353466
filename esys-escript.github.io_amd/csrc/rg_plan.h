// Launch plans: host arithmetic only (no HIP), so that the rules can be
// checked without a device.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <utility>
#include <vector>

namespace rg {

constexpr int kNumXcd = 8;           // MI355X: 8 XCDs, blocks dispatched round-robin
constexpr int kMaxGrid = 8192;       // grid cap of reducing kernels (partials per reduction)
// MI355X's memory-side cache (Infinity Cache, MALL).
constexpr int64_t kMallBytes = 256ll << 20;

// ------------------------------------------- z-marching SpMV (rg_march.h)
constexpr int kMarchThreads = 512;   // nodes of a tile and its ring

struct MarchArgs {
    int n0, n1, n2;
    int tx, ty;          // tile sides
    int gx, gy;          // tiles per plane
    int zs;              // planes per segment
};

// Tiling of a grid of n0 x n1 x n2 nodes for march_block: tiles of at most
// kMarchThreads nodes with their ring, and z segments so that `want`
// workgroups are reached.
inline MarchArgs march_args(int n0, int n1, int n2, int want)
{
    MarchArgs m;
    m.n0 = n0;
    m.n1 = n1;
    m.n2 = n2;
    // least loaded area: nodes plus the ring's share of blocks (9 of 14 along each side)
    double best = 1e300;
    for (int gx = 1; gx <= n0; ++gx) {
        const int tx = (n0 + gx - 1) / gx;
        if (tx + 2 > kMarchThreads / 3 || (n0 + tx - 1) / tx != gx) continue;
        int ty = kMarchThreads / (tx + 2) - 2;
        if (ty < 1) continue;
        if (ty > n1) ty = n1;
        const int gy = (n1 + ty - 1) / ty;
        ty = (n1 + gy - 1) / gy;
        const double area = (double)gx * gy * (tx * ty + 9.0 / 14.0 * (tx + ty));
        if (area < best) {
            best = area;
            m.tx = tx;
            m.ty = ty;
            m.gx = gx;
            m.gy = gy;
        }
    }
    int segs = (int)std::max<int64_t>(1, want / ((int64_t)m.gx * m.gy));
    segs = std::min(segs, std::max(1, n2 / 4));
    m.zs = (n2 + segs - 1) / segs;
    return m;
}
// Tiles x segments, and the workgroups launched for them: a multiple of the
// XCDs, so that xcd_block puts neighbouring tiles, which share the memory
// lines at their edges, on one XCD.
constexpr int64_t march_blocks(const MarchArgs& m) { return (int64_t)m.gx * m.gy * ((m.n2 + m.zs - 1) / m.zs); }
constexpr int64_t march_grid(const MarchArgs& m) { return (march_blocks(m) + kNumXcd - 1) / kNumXcd * kNumXcd; }

// Whether the SpMV of symmetric 3 x 3 blocks marches: values (`bytes`, of
// `vsize` bytes each) that do not fit in the MALL; below that the gather
// kernel's transposed re-reads come from there.  Layered elasticity on n^3
// elements, whole PASO solves gather / march: n = 56 (FP64 values, 187 MB)
// 49.3 / 54.2 ms, 60 (229 MB) 65.9 / 73.7, 64 (277 MB) 94.6 / 87.5, 72
// (392 MB) 134 / 119, 96 (920 MB) 403 / 337; FP32 values 64 (138 MB) 63.1 /
// 67.5, 80 (268 MB) 149 / 125, 96 (460 MB) 280 / 266.
//
// And only where tiles and segments use the chip.  A workgroup takes zs + 1
// steps (planes), each a fixed time (27 barriers) and one per tile node; the
// gather kernel takes a time per node of the grid.  SpMV alone, gather / march
// in us, by N / (steps * (200 + tile nodes)) for FP64 values: 2x2x60000
// elements 11: 192 / 1752, 8x8x9000 70: 251 / 421, 64x63x66 75: 97 / 108,
// 228x228x30 83: 609 / 529, 66^3 85: 104 / 95, 64^3 94: 96 / 88, 96^3 138:
// 301 / 231; tiles of 100 to 144 nodes lose by more than that says (10x10x7000
// 91: 284 / 351, 11x11x5000 100: 245 / 262; 169 nodes, 12x12x4000 108: 238 /
// 223).  FP32 values, whose loads of 40-byte runs and fixed time weigh
// more, by the share of threads with a node, N / (steps * 512 * CUs):
// 8x8x9000 0.15: 129 / 300, 228x228x30 0.39: 331 / 404, 30x30x900 0.41: 164 /
// 202, 260x250x20 0.48: 281 / 265, 200x180x40 0.52: 298 / 265, 96^3 0.58:
// 165 / 155.
//
// Grids with more workgroups than a reduction has partials (some 3.4 M nodes
// per plane) gather too: that kernel's blocks take longer chunks instead.
inline bool march_applies(const MarchArgs& m, int64_t bytes, int vsize, int num_cu)
{
    const int64_t N = (int64_t)m.n0 * m.n1 * m.n2;
    if (N * vsize >= ((int64_t)1 << 32) || bytes <= kMallBytes || march_grid(m) > kMaxGrid) return false;
    if (2 * march_blocks(m) < num_cu) return false;
    const double steps = std::max(1.0, (double)march_blocks(m) / num_cu) * (m.zs + 1) * (num_cu / 256.0);
    return vsize == 8 ? m.tx * m.ty >= 160 && (double)N >= 80.0 * steps * (200 + m.tx * m.ty)
                      : (double)N >= 0.45 * 256 * kMarchThreads * steps;
}

// ------------------------------------------------ assembly (rg_matrix.hip)
// Nodes of a workgroup along each axis and workgroups along each axis.
struct AsmTile {
    int wx = 0, wy = 0, wz = 0;
    int64_t gx = 0, gy = 0, gz = 0;
};
// The wide tile, known to the compiler: npw x 2 x 2 nodes (npw x 4 in 2-D) for
// `npw` nodes per wave and four waves, whose long side reads the coefficients
// in runs.  No tile has more elements around its nodes.
constexpr int asm_wide_y(int dim) { return dim == 3 ? 2 : 4; }
constexpr int asm_wide_z(int dim) { return dim == 3 ? 2 : 1; }
constexpr int asm_tile_elements(int dim, int npw)
{
    return (npw + 1) * (asm_wide_y(dim) + 1) * (dim == 3 ? asm_wide_z(dim) + 1 : 1);
}

// Tile for a grid of nn nodes.  The wide one leaves most threads without a
// node where a grid line has few: there whole lines (wx = nn[0], contiguous in
// memory) and as many of them as fit.  The staged sums of a Brick, whose time
// is that of the workgroups, also take the tile of the fewest workgroups where
// the wide one needs 5/3 as many: sides just over a multiple of npw.  Otherwise
// the wide one is the better although it has idle threads (its index arithmetic
// is the compiler's: two equations 40 -> 60 us with the same tile given at run
// time).  us per call, wide / as here, with C, Y and with A, B, C, D, X, Y on
// quadrature points: one equation on 4x40x60 elements 72 / 38 and 190 / 96,
// 8x8000 28 / 15 and 79 / 37, 64x64x40 154 / 108 and 490 / 318; three equations
// on 7x40x40 93 / 73 and 268 / 188; per element (A, D) 4x40x60 37 / 18.
inline AsmTile asm_tile(int dim, const int64_t* nn, int npw, bool staged)
{
    const int64_t n2 = dim == 3 ? nn[2] : 1;
    const int nodes = 4 * npw, elements = asm_tile_elements(dim, npw);
    auto make = [&](int wx, int wy, int wz) {
        AsmTile t;
        t.wx = wx;
        t.wy = wy;
        t.wz = wz;
        t.gx = (nn[0] + wx - 1) / wx;
        t.gy = (nn[1] + wy - 1) / wy;
        t.gz = (n2 + wz - 1) / wz;
        return t;
    };
    auto count = [](const AsmTile& t) { return t.gx * t.gy * t.gz; };
    const AsmTile wide = make(npw, asm_wide_y(dim), asm_wide_z(dim));
    const bool lines = 2 * nn[0] <= npw;
    if (!lines && (dim == 2 || !staged)) return wide;
    AsmTile best = wide;
    const int from = (int)std::min<int64_t>(nodes, nn[0]);
    for (int wx = from; wx >= (lines ? from : 1); --wx)
        for (int wy = (int)std::min<int64_t>(nodes / wx, nn[1]); wy >= 1; --wy) {
            const int around = (wx + 1) * (wy + 1);
            int wz = 1;
            if (dim == 3) wz = std::min({nodes / (wx * wy), elements / around - 1, (int)std::min<int64_t>(n2, nodes)});
            if (wz < 1 || (dim == 2 && around > elements)) continue;
            const AsmTile t = make(wx, wy, wz);
            if (count(t) < count(best)) best = t;
        }
    return 5 * count(best) < 3 * count(wide) ? best : wide;
}
inline bool asm_is_wide(const AsmTile& t, int dim, int npw)
{
    return t.wx == npw && t.wy == asm_wide_y(dim) && t.wz == asm_wide_z(dim);
}

// --------------------------------------- one-launch solves (rg_resident.hip)
// Tile sides for a grid of n nodes per axis: at most `rows` nodes and
// `cells` padded cells per tile and `tiles` tiles.  Among the shapes that
// fit, the one with the least estimated time per iteration: a reduction over
// G workgroups measured 1.6 / 2.3 / 2.7 / 3.2 / 3.7 / 4.0 us for G = 1 / 8 /
// 32 / 64 / 128 / 256, the stencil about 0.4 us (3-D) or 0.15 us (2-D) per
// 512 rows, a halo of 1024 cells 1.5 us.  With `share` the time counts
// G^share times: 1 for systems that compete for the workgroups.
inline bool resident_tiles(int dim, const int64_t* nn, int rows, int cells, int tiles, int (&t)[3], double share)
{
    const int n[3] = {(int)nn[0], (int)nn[1], dim == 3 ? (int)nn[2] : 1};
    double best = 1e300;
    for (int gz = 1; gz <= std::min(n[2], tiles); ++gz) {
        const int tz = (n[2] + gz - 1) / gz;
        if ((n[2] + tz - 1) / tz != gz) continue;
        for (int gy = 1; gy <= std::min(n[1], tiles / gz); ++gy) {
            const int ty = (n[1] + gy - 1) / gy;
            if ((n[1] + ty - 1) / ty != gy) continue;
            for (int gx = 1; gx <= std::min(n[0], tiles / (gz * gy)); ++gx) {
                const int tx = (n[0] + gx - 1) / gx;
                if ((n[0] + tx - 1) / tx != gx) continue;
                const int64_t vol = (int64_t)tx * ty * tz;
                const int64_t pad = (int64_t)(tx + 2) * (ty + 2) * (dim == 3 ? tz + 2 : 1);
                if (vol > rows || pad > cells) continue;
                const int G = gx * gy * gz;
                double cost = (G > 1 ? 2.0 * (1.4 + 0.3 * std::log2((double)G)) + 1.0 + (pad - vol) / 1024.0 : 1.0) +
                                    (dim == 3 ? 0.4 : 0.15) * (double)((vol + 511) / 512);
                cost *= std::pow((double)G, share);
                if (cost < best) {
                    best = cost;
                    t[0] = tx;
                    t[1] = ty;
                    t[2] = tz;
                }
            }
        }
    }
    return best < 1e300;
}

// Which tiles of which systems each of `blocks` workgroups runs.  Systems go
// in descending order of their expected time (iterations grow with the
// longest side); each takes the workgroups that are free first.  A workgroup
// waits for the others of its system, so every list is in that one order of
// the systems: whatever is sorted or merged here must keep it.
inline void resident_schedule(const std::vector<double>& time, const std::vector<int>& tiles, int blocks,
                              std::vector<int>& first, std::vector<int32_t>& system, std::vector<int32_t>& rank)
{
    std::vector<int> order(time.size()), by_load(blocks);
    for (size_t j = 0; j < order.size(); ++j) order[j] = (int)j;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return time[a] > time[b]; });
    std::vector<double> load(blocks, 0.0);
    std::vector<std::vector<std::pair<int32_t, int32_t>>> list(blocks);
    for (int b = 0; b < blocks; ++b) by_load[b] = b;
    for (int j : order) {
        std::stable_sort(by_load.begin(), by_load.end(), [&](int a, int b) { return load[a] < load[b]; });
        const double end = load[by_load[tiles[j] - 1]] + time[j];
        for (int k = 0; k < tiles[j]; ++k) {
            list[by_load[k]].push_back({(int32_t)j, (int32_t)k});
            load[by_load[k]] = end;
        }
    }
    first.assign(1, 0);
    system.clear();
    rank.clear();
    for (int b = 0; b < blocks; ++b) {
        for (auto& e : list[b]) {
            system.push_back(e.first);
            rank.push_back(e.second);
        }
        first.push_back((int)system.size());
    }
}

}  // namespace rg
