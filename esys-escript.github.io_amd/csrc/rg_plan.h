// Launch plans: host arithmetic only (no HIP), so that the rules can be
// checked without a device.
#pragma once

#include <algorithm>
#include <cstdint>

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
// 67.5, 80 (268 MB) 149 / 125, 96 (460 MB) 280 / 266.  Thin grids without a
// tile for at least every other CU gather.  So do grids with more workgroups
// than a reduction has partials (some 3.4 M nodes per plane; the gather
// kernel's blocks take longer chunks instead).
inline bool march_applies(const MarchArgs& m, int64_t bytes, int vsize, int num_cu)
{
    const int64_t N = (int64_t)m.n0 * m.n1 * m.n2;
    return N * vsize < ((int64_t)1 << 32) && bytes > kMallBytes && 2 * march_blocks(m) >= num_cu &&
           march_grid(m) <= kMaxGrid;
}

}  // namespace rg
