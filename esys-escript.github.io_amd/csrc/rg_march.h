// SpMV of symmetric block stencils by marching in z, each stored block read
// once.
//
// Symmetric storage holds the main and upper blocks; the gather kernels
// (rg_stencil.h) read every upper block again, transposed, for the row below
// it.  For scalar rows those re-reads hit the XCD's L2; for 3 x 3 blocks a
// z-plane of values (97^2 nodes: 9.5 MB) does not fit there, and the SpMV
// moves 1.6 times the stored bytes.  Here a workgroup takes a tile of nodes
// and marches up a z segment: a thread loads a node's blocks once, adds
// A x_j to its own row (registers) and A^T x_i to the row of the neighbour,
// in LDS, which holds the sums of two planes.  Within one slot every thread
// adds to another node, so a barrier between slots keeps the sums free of
// races and their order fixed.  The ring of nodes around the tile is loaded
// too, but only the blocks that reach into the tile (about 7 % more bytes at
// 25 x 14 nodes), and of the plane below the segment those that reach up.
#pragma once

#include "rg_device.h"
#include "rg_plan.h"
#include "rg_stencil.h"

namespace rg {

// Barrier for LDS data: loads from memory stay in flight.
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// epi(node, y, x) for every row of tile and segment `block`, with the row's
// product y and its entries x of the input.
template <int BS, typename VT, class Epi>
__device__ __forceinline__ void march_block(const MarchArgs& g, int block, const VT* __restrict__ val, int64_t ld,
                                            const double* __restrict__ x, Epi&& epi)
{
    constexpr int CEN = StencilShape<3>::CENTER, NST = CEN + 1, B2 = BS * BS;
    __shared__ double X[2][BS][kMarchThreads];   // input, planes z and z + 1
    __shared__ double Q[2][BS][kMarchThreads];   // sums of the transposed products
    const int tid = threadIdx.x;
    const int ew = g.tx + 2;
    const int bx = block % g.gx, by = (block / g.gx) % g.gy, bz = block / (g.gx * g.gy);
    const int ex = tid % ew, ey = tid / ew;
    const int nx = bx * g.tx - 1 + ex, ny = by * g.ty - 1 + ey;
    const bool in = ey < g.ty + 2 && nx >= 0 && nx < g.n0 && ny >= 0 && ny < g.n1;
    auto tile = [&](int cx, int cy) {   // whether cell (cx, cy) is a node of the tile
        return cx >= 1 && cx <= g.tx && cy >= 1 && cy <= g.ty && bx * g.tx - 1 + cx < g.n0 && by * g.ty - 1 + cy < g.n1;
    };
    const bool own = in && tile(ex, ey);
    unsigned reach = 0;                  // bit (dx + 1) + 3 (dy + 1): that neighbour is a node of the tile
#pragma unroll
    for (int d = 0; d < 9; ++d)
        if (in && tile(ex + d % 3 - 1, ey + d / 3 - 1)) reach |= 1u << d;
    const int64_t plane = (int64_t)g.n0 * g.n1, col = nx + (int64_t)g.n0 * ny;
    const int zb = bz * g.zs, ze = min(g.n2, zb + g.zs), z0 = zb > 0 ? zb - 1 : 0;

    // whether this thread uses stored slot t of its node in plane z
    auto needs = [&](int z, int t) {
        if (t == 0) return own && z >= zb;
        const int s = CEN + t, d = s % 9;
        const bool up = s >= 18, hit = (reach >> d) & 1;
        if (z < zb) return up && hit;
        return own || (hit && !(up && z + 1 >= ze));
    };
    // (a 32-bit byte offset of the node beside the stream's base: one register
    // per thread instead of an address pair per stream)
    const uint32_t step = (uint32_t)(plane * sizeof(VT)), off0 = (uint32_t)(col * (int64_t)sizeof(VT));
    auto fetch = [&](int z, int t, VT (&A)[B2]) {
        if (z < ze && needs(z, t)) {
            const uint32_t off = off0 + (uint32_t)z * step;
#pragma unroll
            for (int e = 0; e < B2; ++e)
                A[e] = *reinterpret_cast<const VT*>(reinterpret_cast<const char*>(val + (int64_t)(t * B2 + e) * ld) + off);
        }
    };
    auto load_x = [&](int z, double (&v)[BS]) {
#pragma unroll
        for (int c = 0; c < BS; ++c) v[c] = (in && z < g.n2) ? x[(z * plane + col) * BS + c] : 0.0;
    };
    double v0[BS], v1[BS];
    load_x(z0, v0);
    load_x(z0 + 1, v1);
#pragma unroll
    for (int c = 0; c < BS; ++c) {
        X[z0 & 1][c][tid] = v0[c];
        X[(z0 + 1) & 1][c][tid] = v1[c];
        Q[0][c][tid] = Q[1][c][tid] = 0.0;
    }
    VT A[2][B2];
#pragma unroll
    for (int e = 0; e < B2; ++e) A[0][e] = A[1][e] = (VT)0;
    fetch(z0, 0, A[0]);
    fetch(z0, 1, A[1]);
    for (int z = z0; z < ze; ++z) {
        load_x(z + 2, v1);
        lds_barrier();
        const int cur = z & 1;
        double xi[BS], acc[BS];
#pragma unroll
        for (int c = 0; c < BS; ++c) {
            xi[c] = X[cur][c][tid];
            acc[c] = 0.0;
        }
        const bool mine = own && z >= zb;
#pragma unroll
        for (int t = 0; t < NST; ++t) {
            const int s = CEN + t, d = s % 9, dx = d % 3 - 1, dy = d / 3 - 1, up = s >= 18 ? 1 : 0;
            const int j = tid + dx + ew * dy, pl = cur ^ up;
            const VT(&B)[B2] = A[t & 1];
            if (mine) {
#pragma unroll
                for (int c = 0; c < BS; ++c) {
                    const double xj = t ? X[pl][c][j] : xi[c];
#pragma unroll
                    for (int r = 0; r < BS; ++r) acc[r] = fma((double)B[r + BS * c], xj, acc[r]);
                }
            }
            if (t > 0) {
                const bool hit = ((reach >> d) & 1) && (up ? z + 1 < ze : z >= zb);
                if (hit) {
#pragma unroll
                    for (int c = 0; c < BS; ++c) {
                        double q = Q[pl][c][j];
#pragma unroll
                        for (int r = 0; r < BS; ++r) q = fma((double)B[r + BS * c], xi[r], q);
                        Q[pl][c][j] = q;
                    }
                }
            }
            if (t + 2 < NST) fetch(z, t + 2, A[t & 1]);
            else fetch(z + 1, t + 2 - NST, A[t & 1]);
            if (t > 0) lds_barrier();
        }
        if (mine) {
            double y[BS];
#pragma unroll
            for (int c = 0; c < BS; ++c) y[c] = acc[c] + Q[cur][c][tid];
            epi(z * plane + col, y, xi);
        }
#pragma unroll
        for (int c = 0; c < BS; ++c) {
            Q[cur][c][tid] = 0.0;
            X[cur][c][tid] = v1[c];
        }
    }
}

}  // namespace rg
