// Krylov solves of small scalar systems in one launch.
//
// A matrix of a few hundred thousand rows fits in the chip's registers: every
// workgroup owns one brick of nodes (a tile), keeps the full stencil rows of
// its nodes and all its Krylov vectors in registers, and the vector the
// operator is applied to in LDS with one layer of halo cells.  What crosses
// workgroups goes through memory past the L2s (relaxed agent-scope accesses,
// written through and read through): the surface values of the tiles and, per
// reduction, one slot of partial sums per workgroup.
//
// A reduction is also the barrier: each workgroup stores its sums into its
// slot and reads every slot until none is empty, in the same order, so all
// get the same totals.  Slots hold kEmpty until written; there are four sets
// of them, and a workgroup empties its slot of the set after next once it has
// passed a reduction: all others have then finished with it, and it is empty
// again before any of them can look.  The surface values are stored (and
// waited for) before the slot is written, so whoever has seen all slots reads
// the neighbours' values of this step.
//
// Bound: latency.  The launch sequence it replaces spends 2-5 us per kernel
// on boundaries and 6 (PASO PCG) to 13 (BiCGStab) kernels per iteration;
// here an iteration is two (three for BiCGStab) reductions of 2-4 us.  Whole
// solves with set-up, launch sequence -> here: PASO PCG Rectangle 256^2 19.4
// -> 6.2 ms (7 us per iteration), Brick 61x47x53 10.2 -> 3.5 ms, Rectangle
// 20x13 2.26 -> 0.50 ms; BiCGStab Brick 63x64x40 24.6 -> 5.5 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <utility>
#include <vector>

#include "rg_device.h"
#include "rg_plan.h"
#include "rg_resident.h"
#include "rg_stencil.h"

namespace rg {

namespace {

constexpr int kResThreads = 512;   // two waves per SIMD, 256 registers each
constexpr int kResWaves = kResThreads / 64;
constexpr int kMaxSums = 4;        // sums of one reduction
constexpr int kSets = 4;           // sets of slots
constexpr int kMaxTiles = 256;     // one per CU
// An empty slot: a denormal (about 1e-309; a sum of these very bits is stored
// as its neighbour).  A finite number, because freed slots become other
// buffers' uninitialised memory.
constexpr unsigned long long kEmpty = 0x0000DEADBEEF0001ull;

// One system: its matrix, grid and tiling.
struct ResSystem {
    const double* val;
    const double* dinv;
    int64_t ld;
    int n0, n1, n2;
    int tx, ty, tz;      // tile sides
    int gx, gy, gz;      // tiles per axis
    int sym;
};

struct ResArgs {
    ResSystem sys;
    const double* r;
    double* x;
    double* pub0;        // surface values by node
    double* pub1;
    double* pub2;
    unsigned long long* slots;
    KrylovState* st;
    int maxit;
    unsigned spins;
    double tol;
};

__device__ __forceinline__ void put(unsigned long long* p, unsigned long long v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long get(const unsigned long long* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void put(double* p, double v)
{
    put(reinterpret_cast<unsigned long long*>(p), (unsigned long long)__double_as_longlong(v));
}
__device__ __forceinline__ double get(const double* p)
{
    return __longlong_as_double((long long)get(reinterpret_cast<const unsigned long long*>(p)));
}

// Sum over a wave by row shifts and row broadcasts (register moves; the
// ds_bpermute butterfly of wave_sum takes four times as long and sits on the
// critical path of every reduction here); all lanes get it.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, true);
    return v + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double wave_total(double v)
{
    v = dpp_add<0x111, 0xf>(v);   // row_shr:1, 2, 4, 8: lane 15 of each row of 16 holds its sum
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    v = dpp_add<0x118, 0xf>(v);
    v = dpp_add<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
    v = dpp_add<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, 63), hi = __builtin_amdgcn_readlane((int)(b >> 32), 63);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

struct ResShared {
    double red[kMaxSums][kResWaves];
    double tot[kMaxSums];
    int bad;
};

// The workgroups that solve one system: this one's rank among them and their
// slots, kSets x size x kMaxSums.
struct Gang {
    unsigned long long* slots;
    int size, rank;
    unsigned spins;      // polls of the slots before a workgroup gives up
};

// Totals of v over the gang (valid in all threads, the same bits in all
// workgroups); false once a workgroup has waited too long, whereupon every
// workgroup of the gang ends.
template <int NV>
__device__ __forceinline__ bool reduce_all(ResShared& sh, const Gang& a, unsigned& epoch, double (&v)[NV])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, G = a.size;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const double s = wave_total(v[k]);
        if (lane == 0) sh.red[k][w] = s;
    }
    // A workgroup barrier with a full wait between its fence and itself: this
    // wave's surface values and emptied slots are issued before the fence and
    // have arrived before any slot is written (the fence alone lets agent-scope
    // stores be in flight, and the wait by itself does not name memory).  As an
    // asm with a memory clobber, before or behind the sums, it cost single
    // methods 0.5 to 2 %.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (w == 0) {
        double s[NV];
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            s[k] = sh.red[k][0];
#pragma unroll
            for (int j = 1; j < kResWaves; ++j) s[k] += sh.red[k][j];
        }
        bool miss = false;
        if (G > 1) {
            unsigned long long* cur = a.slots + (size_t)(epoch & (kSets - 1)) * G * kMaxSums;
            unsigned long long* nxt = a.slots + (size_t)((epoch + 2) & (kSets - 1)) * G * kMaxSums;
#pragma unroll
            for (int k = 0; k < NV; ++k)
                if (lane == k) {
                    const unsigned long long b = (unsigned long long)__double_as_longlong(s[k]);
                    put(cur + a.rank * kMaxSums + k, b == kEmpty ? b ^ 1 : b);
                }
            unsigned long long u[kMaxTiles / 64][NV];
            unsigned left = a.spins;
            do {
                miss = false;
#pragma unroll
                for (int j = 0; j < kMaxTiles / 64; ++j) {
                    const int g = lane + 64 * j;
#pragma unroll
                    for (int k = 0; k < NV; ++k) u[j][k] = g < G ? get(cur + g * kMaxSums + k) : 0ull;
                }
#pragma unroll
                for (int j = 0; j < kMaxTiles / 64; ++j)
#pragma unroll
                    for (int k = 0; k < NV; ++k) miss = miss || u[j][k] == kEmpty;
                miss = __any(miss);
            } while (miss && --left > 0);
            if (lane < kMaxSums) put(nxt + a.rank * kMaxSums + lane, kEmpty);
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                double t = __longlong_as_double((long long)u[0][k]);
#pragma unroll
                for (int j = 1; j < kMaxTiles / 64; ++j) t += __longlong_as_double((long long)u[j][k]);
                s[k] = wave_total(t);
            }
        }
        if (lane == 0) {
#pragma unroll
            for (int k = 0; k < NV; ++k) sh.tot[k] = s[k];
            sh.bad = miss;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = sh.tot[k];
    ++epoch;
    return !sh.bad;
}

// Rows per thread: as many as leave the stencil rows and the method's vectors
// in 256 registers (k_resident<3, PCG> spills two of them and
// k_resident_batch<3> four; a row less would cut the systems that fit by a third).
template <int DIM, int METHOD>
__host__ __device__ constexpr int res_rows()
{
    return DIM == 2 ? (METHOD == RG_METHOD_BICGSTAB ? 3 : 4) : (METHOD == RG_METHOD_PCG || METHOD == RG_METHOD_PCG_PLAIN) ? 3 : 2;
}
// Padded tile cells per thread.
template <int DIM, int METHOD>
__host__ __device__ constexpr int res_cells()
{
    return res_rows<DIM, METHOD>() + 3;
}

// One tile's rows in the registers of a workgroup, M per thread, and the
// padded cells it reads of other tiles, KH per thread.
template <int DIM, int M, int KH>
struct ResTile {
    static constexpr int NS = StencilShape<DIM>::NS;
    int px, py;          // padded sides
    int halo[KH];        // node of padded cell tid + k * threads; -1: the tile's own, or outside the grid
    int node[M];         // own rows; -1: outside the tile's part of the grid (zero stencil, reads cell (1, 1, 1))
    int cell[M];         // padded cell
    bool surf[M];        // on the tile's surface
    double A[M][NS], di[M];

    // Indices are made opaque at each use: kept over the iterations, the
    // addresses formed from them took some 60 registers.
    static __device__ __forceinline__ int opaque(int i)
    {
        asm volatile("" : "+v"(i));
        return i;
    }
    // Padded cells of a tile of system s.
    static __host__ __device__ __forceinline__ int cells(const ResSystem& s)
    {
        return (s.tx + 2) * (s.ty + 2) * (DIM == 3 ? s.tz + 2 : 1);
    }

    __device__ __forceinline__ void setup(const ResSystem& s, int rank, int gang)
    {
        constexpr int CEN = StencilShape<DIM>::CENTER;
        const int tid = threadIdx.x;
        px = s.tx + 2;
        py = s.ty + 2;
        const int total = cells(s);
        const int x0 = rank % s.gx * s.tx, y0 = (rank / s.gx) % s.gy * s.ty, z0 = rank / (s.gx * s.gy) * s.tz;
        const int s1 = s.n0, s2 = s.n0 * s.n1;
#pragma unroll
        for (int k = 0; k < KH; ++k) {
            const int c = tid + k * kResThreads;
            halo[k] = -1;
            if (c < total) {
                const int cx = c % px, cy = (c / px) % py, cz = DIM == 3 ? c / (px * py) : 1;
                const int gx = x0 + cx - 1, gy = y0 + cy - 1, gz = DIM == 3 ? z0 + cz - 1 : 0;
                const bool own = cx >= 1 && cx <= s.tx && cy >= 1 && cy <= s.ty && (DIM == 2 || (cz >= 1 && cz <= s.tz));
                const bool in = gx >= 0 && gx < s.n0 && gy >= 0 && gy < s.n1 && gz >= 0 && gz < s.n2;
                if (!own && in) halo[k] = gx + s1 * gy + s2 * gz;
            }
        }
        const int tile = s.tx * s.ty * (DIM == 3 ? s.tz : 1);
#pragma unroll
        for (int j = 0; j < M; ++j) {
            const int l = tid + j * kResThreads;
            const int lx = l % s.tx, ly = (l / s.tx) % s.ty, lz = DIM == 3 ? l / (s.tx * s.ty) : 0;
            const bool in = l < tile && x0 + lx < s.n0 && y0 + ly < s.n1 && (DIM == 2 || z0 + lz < s.n2);
            node[j] = in ? (x0 + lx) + s1 * (y0 + ly) + s2 * (DIM == 3 ? z0 + lz : 0) : -1;
            cell[j] = in ? (lx + 1) + px * ((ly + 1) + (DIM == 3 ? py * (lz + 1) : 0))
                         : 1 + px * (1 + (DIM == 3 ? py : 0));
            surf[j] = in && gang > 1 && (lx == 0 || lx == s.tx - 1 || ly == 0 || ly == s.ty - 1 ||
                                         (DIM == 3 && (lz == 0 || lz == s.tz - 1)));
            const int i = in ? node[j] : 0;
            di[j] = in ? s.dinv[i] : 0.0;
#pragma unroll
            for (int q = 0; q < NS; ++q) {
                int dx, dy, dz;
                slot_delta<DIM>(q, dx, dy, dz);
                double v;
                if (!s.sym) {
                    v = s.val[(int64_t)q * s.ld + i];
                } else if (q >= CEN) {
                    v = s.val[(int64_t)(q - CEN) * s.ld + i];
                } else {
                    const int jn = i + dx + dy * s1 + dz * s2;
                    v = jn >= 0 ? s.val[(int64_t)(CEN - q) * s.ld + jn] : 0.0;
                }
                A[j][q] = in ? v : 0.0;
            }
        }
    }
    __device__ __forceinline__ double apply(const double* V, int j) const
    {
        double acc = 0.0;
        const double* c = V + opaque(cell[j]);
#pragma unroll
        for (int q = 0; q < NS; ++q) {
            int dx, dy, dz;
            slot_delta<DIM>(q, dx, dy, dz);
            acc = fma(A[j][q], c[dx + px * (dy + py * dz)], acc);
        }
        __builtin_amdgcn_sched_barrier(0);   // one row's loads in flight at a time: registers
        return acc;
    }
    __device__ __forceinline__ void publish(double* pub, int j, double v) const
    {
        if (surf[j]) put(pub + opaque(node[j]), v);
    }
    __device__ __forceinline__ void own(double* V, int j, double v) const
    {
        if (node[j] >= 0) V[cell[j]] = v;
    }
    __device__ __forceinline__ double neighbour(const double* pub, int k) const
    {
        return halo[k] >= 0 ? get(pub + opaque(halo[k])) : 0.0;
    }
};

// The recurrences are those of the launch sequences (stage_apply and the
// update kernels of the solver): PASO's residual-smoothed PCG, the textbook
// PCG, BiCGStab and MINRES with one Jacobi sweep, and the same stopping
// tests in the same order.
template <int DIM, int METHOD>
__global__ __launch_bounds__(kResThreads) void k_resident(ResArgs a)
{
    constexpr int M = res_rows<DIM, METHOD>();
    constexpr int KH = res_cells<DIM, METHOD>();
    constexpr bool BICG = METHOD == RG_METHOD_BICGSTAB;
    __shared__ ResShared sh;
    extern __shared__ double lds[];
    const int tid = threadIdx.x;
    const Gang gang{a.slots, (int)gridDim.x, (int)blockIdx.x, a.spins};
    ResTile<DIM, M, KH> T;
    T.setup(a.sys, gang.rank, gang.size);
    const auto& node = T.node;
    const auto& cell = T.cell;
    const auto& halo = T.halo;
    const auto& di = T.di;
    const int cells = T.cells(a.sys);
    double* P = lds;             // the vector the operator is applied to
    double* S = lds + cells;     // BiCGStab: the second one
    double* X = lds + (BICG ? 2 : 1) * cells + tid;   // the iterate of this thread's rows
    double* X2 = X + M * kResThreads;                 // PASO: the unsmoothed one
    for (int c = tid; c < (BICG ? 2 : 1) * cells; c += kResThreads) lds[c] = 0.0;
    __syncthreads();
    double r[M];
#pragma unroll
    for (int j = 0; j < M; ++j) {
        r[j] = node[j] >= 0 ? a.r[node[j]] : 0.0;
        X[j * kResThreads] = node[j] >= 0 ? a.x[node[j]] : 0.0;
    }

    unsigned epoch = 0;
    int status = KS_RUNNING, iter = 0;
    double norm = 0.0;
    bool ok = true;

    if constexpr (METHOD == RG_METHOD_PCG || METHOD == RG_METHOD_PCG_PLAIN) {
        constexpr bool PASO = METHOD == RG_METHOD_PCG;
        double rs[PASO ? M : 1];
        double beta = 0.0, rho;
        {
            double t[2] = {0.0, 0.0};
#pragma unroll
            for (int j = 0; j < M; ++j) {
                const double z = di[j] * r[j];
                T.publish(a.pub0, j, z);
                t[0] = fma(z, r[j], t[0]);
                t[1] = fma(r[j], r[j], t[1]);
                if constexpr (PASO) {
                    rs[j] = r[j];
                    X2[j * kResThreads] = X[j * kResThreads];
                }
            }
            ok = reduce_all<2>(sh, gang, epoch, t);
            rho = t[0];
            if constexpr (PASO) {
                iter = 1;
            } else {
                norm = sqrt(t[1]);
                if (norm <= a.tol) status = KS_CONVERGED;
                else if (a.maxit <= 0) status = KS_MAXITER;
                else if (fabs(rho) <= 0.0) status = KS_BREAKDOWN;
            }
        }
        while (ok && status == KS_RUNNING) {
            // p = z + beta p, also in the halo
            double zh[KH];
#pragma unroll
            for (int k = 0; k < KH; ++k) zh[k] = T.neighbour(a.pub0, k);
#pragma unroll
            for (int j = 0; j < M; ++j) T.own(P, j, fma(beta, P[cell[j]], di[j] * r[j]));
#pragma unroll
            for (int k = 0; k < KH; ++k)
                if (halo[k] >= 0) P[tid + k * kResThreads] = fma(beta, P[tid + k * kResThreads], zh[k]);
            __syncthreads();
            double q[M], d[1] = {0.0};
#pragma unroll
            for (int j = 0; j < M; ++j) {
                q[j] = T.apply(P, j);
                d[0] = fma(q[j], P[cell[j]], d[0]);
            }
            ok = reduce_all<1>(sh, gang, epoch, d);
            if (!ok) break;
            if (fabs(d[0]) <= 0.0) {
                status = KS_BREAKDOWN;
                break;
            }
            const double alpha = rho / d[0];
            if constexpr (!PASO) {
                double t[2] = {0.0, 0.0};
#pragma unroll
                for (int j = 0; j < M; ++j) {
                    r[j] = fma(-alpha, q[j], r[j]);
                    const double z = di[j] * r[j];
                    T.publish(a.pub0, j, z);
                    t[0] = fma(z, r[j], t[0]);
                    t[1] = fma(r[j], r[j], t[1]);
                }
#pragma unroll
                for (int j = 0; j < M; ++j)
                    X[j * kResThreads] = fma(alpha, P[cell[j]], X[j * kResThreads]);
                ok = reduce_all<2>(sh, gang, epoch, t);
                if (!ok) break;
                ++iter;
                norm = sqrt(t[1]);
                if (norm <= a.tol) status = KS_CONVERGED;
                else if (iter >= a.maxit) status = KS_MAXITER;
                else if (fabs(t[0]) <= 0.0) status = KS_BREAKDOWN;
                beta = t[0] / rho;
                rho = t[0];
            } else {
                // d = r - rs, s3 = d.d, s4 = d.rs, rs.rs, and the next r.z
                double t[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int j = 0; j < M; ++j) {
                    r[j] = fma(-alpha, q[j], r[j]);
                    const double z = di[j] * r[j];
                    T.publish(a.pub0, j, z);
                    const double e = r[j] - rs[j];
                    t[0] = fma(e, e, t[0]);
                    t[1] = fma(e, rs[j], t[1]);
                    t[2] = fma(rs[j], rs[j], t[2]);
                    t[3] = fma(z, r[j], t[3]);
                    X2[j * kResThreads] = fma(alpha, P[cell[j]], X2[j * kResThreads]);
                }
                ok = reduce_all<4>(sh, gang, epoch, t);
                if (!ok) break;
                const double g1 = fabs(t[0]) <= 0.0 ? 0.0 : -t[1] / t[0], g2 = 1.0 - g1;
                double nn[1] = {0.0};
#pragma unroll
                for (int j = 0; j < M; ++j) {
                    rs[j] = g2 * rs[j] + g1 * r[j];
                    X[j * kResThreads] = g2 * X[j * kResThreads] + g1 * X2[j * kResThreads];
                    nn[0] = fma(rs[j], rs[j], nn[0]);
                }
                // ||rs||^2 of the new rs = rs + g1 d from the sums at hand;
                // summed afresh where the step took it so far down that the
                // difference has lost its digits
                norm = t[2] + g1 * (2.0 * t[1] + g1 * t[0]);
                if (!(norm > 1e-4 * t[2])) {
                    ok = reduce_all<1>(sh, gang, epoch, nn);
                    if (!ok) break;
                    norm = nn[0];
                }
                norm = sqrt(norm);
                const bool conv = norm <= a.tol, maxi = iter > a.maxit, brk = fabs(rho) <= 0.0;
                if (conv || maxi || brk) {
                    status = maxi ? KS_MAXITER : (brk ? KS_BREAKDOWN : KS_CONVERGED);
                } else {
                    beta = t[3] / rho;
                    rho = t[3];
                    ++iter;
                }
            }
        }
    } else if constexpr (METHOD == RG_METHOD_MINRES) {
        double ro[M], w[M], wo[M];
        double c = 1.0, co = 1.0, s = 0.0, so = 0.0, gam = 0.0, gold = 0.0, eta = 0.0, tol = a.tol;
        {
            double t[2] = {0.0, 0.0};
#pragma unroll
            for (int j = 0; j < M; ++j) {
                ro[j] = w[j] = wo[j] = 0.0;
                const double z = di[j] * r[j];
                T.publish(a.pub0, j, z);
                t[0] = fma(r[j], z, t[0]);
                t[1] = fma(r[j], r[j], t[1]);
            }
            ok = reduce_all<2>(sh, gang, epoch, t);
            norm = 1.0;
            if (t[0] < 0.0) status = KS_NEGATIVE;
            else if (fabs(t[0]) <= 0.0) status = KS_CONVERGED;
            else if (a.maxit <= 0) status = KS_MAXITER;
            else {
                gam = sqrt(t[0]);
                eta = gam;
                norm = gam;
                tol = a.tol * (gam / sqrt(t[1]));
            }
        }
        while (ok && status == KS_RUNNING) {
            // P = z / gamma, also in the halo
            const double ig = 1.0 / gam;
            double zh[KH];
#pragma unroll
            for (int k = 0; k < KH; ++k) zh[k] = T.neighbour(a.pub0, k);
#pragma unroll
            for (int j = 0; j < M; ++j) T.own(P, j, ig * (di[j] * r[j]));
#pragma unroll
            for (int k = 0; k < KH; ++k)
                if (halo[k] >= 0) P[tid + k * kResThreads] = ig * zh[k];
            __syncthreads();
            double q[M], d[1] = {0.0};
#pragma unroll
            for (int j = 0; j < M; ++j) {
                q[j] = T.apply(P, j);
                d[0] = fma(q[j], P[cell[j]], d[0]);
            }
            ok = reduce_all<1>(sh, gang, epoch, d);
            if (!ok) break;
            const double delta = d[0], f1 = delta / gam, f2 = iter > 0 ? gam / gold : 0.0;
            double t[1] = {0.0};
#pragma unroll
            for (int j = 0; j < M; ++j) {
                double v = fma(-f1, r[j], q[j]);
                if (iter > 0) v = fma(-f2, ro[j], v);
                ro[j] = r[j];
                r[j] = v;
                const double z = di[j] * v;
                T.publish(a.pub0, j, z);
                t[0] = fma(v, z, t[0]);
            }
            ok = reduce_all<1>(sh, gang, epoch, t);
            if (!ok) break;
            if (t[0] < 0.0) status = KS_NEGATIVE;
            else if (fabs(t[0]) <= 0.0) status = KS_CONVERGED;
            else {
                const double gn = sqrt(t[0]);
                const double a0 = c * delta - co * s * gam, a1 = sqrt(a0 * a0 + gn * gn);
                const double a2 = s * delta + co * c * gam, a3 = so * gam, ia1 = 1.0 / a1;
                co = c;
                so = s;
                c = a0 / a1;
                s = gn / a1;
                gold = gam;
                gam = gn;
                norm = norm * s;
                const double ceta = c * eta;
                eta = -s * eta;
#pragma unroll
                for (int j = 0; j < M; ++j) {
                    double v = P[cell[j]];
                    if (iter > 1) v = fma(-a3, wo[j], v);
                    if (iter > 0) v = fma(-a2, w[j], v);
                    wo[j] = w[j];
                    v *= ia1;
                    w[j] = v;
                    X[j * kResThreads] = fma(ceta, v, X[j * kResThreads]);
                }
                if (norm <= tol) status = KS_CONVERGED;
            }
            ++iter;
            if (status == KS_RUNNING && iter >= a.maxit) status = KS_MAXITER;
        }
    } else {
        // BiCGStab.  pub0 / pub1: M^-1 r and M^-1 (p - omega v) of the tile
        // surfaces, from which the halo of phat = M^-1 p follows once beta is
        // known; pub2: M^-1 v, from which the halo of shat follows once alpha
        // is; S holds M^-1 r, then shat = M^-1 s in the halo.  ||s|| is
        // reduced with t.s and t.t (t is not used if it ends the solve).
        double rt[M], p[M], v[M];
        double tau = 0.0, told = 0.0, alpha = 0.0, omega = 0.0;
        {
            double t[1] = {0.0};
#pragma unroll
            for (int j = 0; j < M; ++j) {
                rt[j] = r[j];
                p[j] = v[j] = 0.0;
                T.publish(a.pub0, j, di[j] * r[j]);
                T.publish(a.pub1, j, 0.0);
                t[0] = fma(rt[j], r[j], t[0]);
            }
            ok = reduce_all<1>(sh, gang, epoch, t);
            tau = t[0];
        }
        while (ok) {
            ++iter;
            if (fabs(tau) <= 0.0) {
                status = KS_BREAKDOWN;
                break;
            }
            const double beta = iter > 1 ? tau / told * (alpha / omega) : 0.0;
            double h0[KH], h1[KH];
#pragma unroll
            for (int k = 0; k < KH; ++k) {
                h0[k] = T.neighbour(a.pub0, k);
                h1[k] = T.neighbour(a.pub1, k);
            }
#pragma unroll
            for (int j = 0; j < M; ++j) {
                p[j] = iter > 1 ? r[j] + beta * (p[j] - omega * v[j]) : r[j];
                T.own(P, j, di[j] * p[j]);
            }
#pragma unroll
            for (int k = 0; k < KH; ++k)
                if (halo[k] >= 0) {
                    P[tid + k * kResThreads] = fma(beta, h1[k], h0[k]);
                    S[tid + k * kResThreads] = h0[k];
                }
            __syncthreads();
            double d[1] = {0.0};
#pragma unroll
            for (int j = 0; j < M; ++j) {
                v[j] = T.apply(P, j);
                T.publish(a.pub2, j, di[j] * v[j]);
                d[0] = fma(rt[j], v[j], d[0]);
            }
            ok = reduce_all<1>(sh, gang, epoch, d);
            if (!ok) break;
            if (fabs(d[0]) <= 0.0) {
                status = KS_BREAKDOWN;
                break;
            }
            alpha = tau / d[0];
#pragma unroll
            for (int k = 0; k < KH; ++k) h0[k] = T.neighbour(a.pub2, k);
            double t[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int j = 0; j < M; ++j) {
                r[j] = fma(-alpha, v[j], r[j]);
                T.own(S, j, di[j] * r[j]);
                t[2] = fma(r[j], r[j], t[2]);
            }
#pragma unroll
            for (int k = 0; k < KH; ++k)
                if (halo[k] >= 0) S[tid + k * kResThreads] = fma(-alpha, h0[k], S[tid + k * kResThreads]);
            __syncthreads();
            double tv[M];
#pragma unroll
            for (int j = 0; j < M; ++j) {
                tv[j] = T.apply(S, j);
                t[0] = fma(tv[j], r[j], t[0]);
                t[1] = fma(tv[j], tv[j], t[1]);
            }
            ok = reduce_all<3>(sh, gang, epoch, t);
            if (!ok) break;
            norm = sqrt(t[2]);
            if (norm <= a.tol) {
#pragma unroll
                for (int j = 0; j < M; ++j)
                    X[j * kResThreads] = fma(alpha, P[cell[j]], X[j * kResThreads]);
                status = KS_CONVERGED;
                break;
            }
            if (fabs(t[1]) <= 0.0) {
                status = KS_BREAKDOWN;
                break;
            }
            omega = t[0] / t[1];
            double e[2] = {0.0, 0.0};
#pragma unroll
            for (int j = 0; j < M; ++j) {
                X[j * kResThreads] += alpha * P[cell[j]] + omega * S[cell[j]];
                r[j] = fma(-omega, tv[j], r[j]);
                T.publish(a.pub0, j, di[j] * r[j]);
                T.publish(a.pub1, j, di[j] * (p[j] - omega * v[j]));
                e[0] = fma(r[j], r[j], e[0]);
                e[1] = fma(rt[j], r[j], e[1]);
            }
            ok = reduce_all<2>(sh, gang, epoch, e);
            if (!ok) break;
            norm = sqrt(e[0]);
            const bool conv = norm <= a.tol, maxi = iter > a.maxit, brk = fabs(omega) <= 0.0;
            if (conv || maxi || brk) {
                status = maxi ? KS_MAXITER : (brk ? KS_BREAKDOWN : KS_CONVERGED);
                break;
            }
            told = tau;
            tau = e[1];
        }
    }
    if (ok) {
#pragma unroll
        for (int j = 0; j < M; ++j)
            if (node[j] >= 0) a.x[node[j]] = X[j * kResThreads];
    } else if (tid == 0) {
        a.st->gave_up = 1;
    }
    if (ok && gang.rank == 0 && tid == 0) {
        a.st->status = status;
        a.st->num_iter = iter;
        a.st->norm = norm;
        a.st->done = 1;
    }
}

// Textbook Jacobi-PCG of many independent systems from x = 0 (unbalanced).
// Workgroup b runs its tasks, one tile of one system each, in order; the
// workgroups of a system form a gang.  All workgroups are resident and every
// list is in the one order of all systems that resident_schedule takes them in,
// so the earliest unfinished system of that order always has all its
// workgroups at work.  24 Rectangles n ~ U{64..400} (1.4 M rows,
// 3000 iterations of the largest): 121 ms in five launches per iteration over
// all systems -> 33 ms.
struct ResBatchSystem {
    ResSystem sys;
    const double* b;
    double* x;
    double* pub0;
    double* pub1;
    unsigned long long* slots;
};
struct ResTask {
    int32_t system, rank;
};
struct ResBatchArgs {
    const ResBatchSystem* systems;
    const ResTask* tasks;
    const int* first;            // tasks of workgroup b: first[b] .. first[b + 1]
    KrylovState* st;
    int maxit;
    unsigned spins;
    double tol;                  // relative
};

constexpr int kBatchRows2 = 6, kBatchRows3 = 3;   // rows per thread, 2-D and 3-D
// The recursive residual is taken this far below the tolerance before
// b - A x is looked at: the launch sequence looks every 32 iterations and so
// goes past the tolerance by up to as many, and its callers have solutions
// that accurate (about 8 % more iterations than stopping at the tolerance).
constexpr double kBatchMargin = 0.1;

template <int DIM>
__global__ __launch_bounds__(kResThreads) void k_resident_batch(ResBatchArgs a)
{
    constexpr int M = DIM == 2 ? kBatchRows2 : kBatchRows3, KH = M + 3;
    __shared__ ResShared sh;
    extern __shared__ double lds[];
    const int tid = threadIdx.x;
    for (int task = a.first[blockIdx.x]; task < a.first[blockIdx.x + 1]; ++task) {
        const ResBatchSystem B = a.systems[a.tasks[task].system];
        const Gang gang{B.slots, B.sys.gx * B.sys.gy * B.sys.gz, a.tasks[task].rank, a.spins};
        KrylovState* st = a.st + a.tasks[task].system;
        ResTile<DIM, M, KH> T;
        T.setup(B.sys, gang.rank, gang.size);
        const int cells = T.cells(B.sys);
        double* P = lds;
        double* X = lds + cells + tid;
        __syncthreads();         // the previous task's last reads
        for (int c = tid; c < cells; c += kResThreads) P[c] = 0.0;
        __syncthreads();
        unsigned epoch = 0;
        int status = KS_RUNNING, iter = 0;
        double norm, beta = 0.0, rho, tol;
        double r[M], t[2] = {0.0, 0.0};
#pragma unroll
        for (int j = 0; j < M; ++j) {
            r[j] = T.node[j] >= 0 ? B.b[T.node[j]] : 0.0;
            X[j * kResThreads] = 0.0;
            const double z = T.di[j] * r[j];
            T.publish(B.pub0, j, z);
            t[0] = fma(z, r[j], t[0]);
            t[1] = fma(r[j], r[j], t[1]);
        }
        bool ok = reduce_all<2>(sh, gang, epoch, t);
        rho = t[0];
        norm = sqrt(t[1]);
        tol = a.tol * norm;
        if (norm <= tol) status = KS_CONVERGED;
        else if (a.maxit <= 0) status = KS_MAXITER;
        else if (fabs(rho) <= 0.0) status = KS_BREAKDOWN;
        while (ok && status == KS_RUNNING) {
            double zh[KH];
#pragma unroll
            for (int k = 0; k < KH; ++k) zh[k] = T.neighbour(B.pub0, k);
#pragma unroll
            for (int j = 0; j < M; ++j) T.own(P, j, fma(beta, P[T.cell[j]], T.di[j] * r[j]));
#pragma unroll
            for (int k = 0; k < KH; ++k)
                if (T.halo[k] >= 0) P[tid + k * kResThreads] = fma(beta, P[tid + k * kResThreads], zh[k]);
            __syncthreads();
            double q[M], d[1] = {0.0};
#pragma unroll
            for (int j = 0; j < M; ++j) {
                q[j] = T.apply(P, j);
                d[0] = fma(q[j], P[T.cell[j]], d[0]);
            }
            ok = reduce_all<1>(sh, gang, epoch, d);
            if (!ok) break;
            if (fabs(d[0]) <= 0.0) {
                status = KS_BREAKDOWN;
                break;
            }
            const double alpha = rho / d[0];
            t[0] = t[1] = 0.0;
#pragma unroll
            for (int j = 0; j < M; ++j) {
                r[j] = fma(-alpha, q[j], r[j]);
                X[j * kResThreads] = fma(alpha, P[T.cell[j]], X[j * kResThreads]);
                const double z = T.di[j] * r[j];
                T.publish(B.pub0, j, z);
                t[0] = fma(z, r[j], t[0]);
                t[1] = fma(r[j], r[j], t[1]);
            }
            ok = reduce_all<2>(sh, gang, epoch, t);
            if (!ok) break;
            ++iter;
            norm = sqrt(t[1]);
            beta = t[0] / rho;
            rho = t[0];
            const bool maxi = iter >= a.maxit;
            if (norm <= kBatchMargin * tol || (maxi && norm <= tol)) {
                // r = b - A x decides (x goes through P; the search starts
                // again from the new residual if it does not end here)
                double one[1] = {0.0};
#pragma unroll
                for (int j = 0; j < M; ++j) T.publish(B.pub1, j, X[j * kResThreads]);
                ok = reduce_all<1>(sh, gang, epoch, one);
                if (!ok) break;
#pragma unroll
                for (int k = 0; k < KH; ++k) zh[k] = T.neighbour(B.pub1, k);
#pragma unroll
                for (int j = 0; j < M; ++j) T.own(P, j, X[j * kResThreads]);
#pragma unroll
                for (int k = 0; k < KH; ++k)
                    if (T.halo[k] >= 0) P[tid + k * kResThreads] = zh[k];
                __syncthreads();
                t[0] = t[1] = 0.0;
#pragma unroll
                for (int j = 0; j < M; ++j) {
                    r[j] = (T.node[j] >= 0 ? B.b[T.node[j]] : 0.0) - T.apply(P, j);
                    if (T.node[j] < 0) r[j] = 0.0;
                    const double z = T.di[j] * r[j];
                    T.publish(B.pub0, j, z);
                    t[0] = fma(z, r[j], t[0]);
                    t[1] = fma(r[j], r[j], t[1]);
                }
                ok = reduce_all<2>(sh, gang, epoch, t);
                if (!ok) break;
                norm = sqrt(t[1]);
                rho = t[0];
                beta = 0.0;
                if (norm <= tol) {
                    status = KS_CONVERGED;
                    break;
                }
            }
            if (maxi) status = KS_MAXITER;
            else if (fabs(rho) <= 0.0) status = KS_BREAKDOWN;
        }
        if (ok) {
#pragma unroll
            for (int j = 0; j < M; ++j)
                if (T.node[j] >= 0) B.x[T.node[j]] = X[j * kResThreads];
        } else if (tid == 0) {
            st->gave_up = 1;
        }
        if (ok && gang.rank == 0 && tid == 0) {
            st->status = status;
            st->num_iter = iter;
            st->norm = norm;
            st->done = 1;
        }
    }
}

__global__ void k_res_empty(unsigned long long* slots, int64_t nslots, KrylovState* st, int count)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (int64_t i = t; i < nslots; i += (int64_t)gridDim.x * blockDim.x) slots[i] = kEmpty;
    for (int64_t i = t; i < count; i += (int64_t)gridDim.x * blockDim.x) {
        st[i].done = 0;
        st[i].status = KS_RUNNING;
        st[i].num_iter = 0;
        st[i].norm = 0.0;
        st[i].gave_up = 0;
    }
}

template <class F>
bool by_method(int dim, int method, F&& f)
{
    auto go = [&](auto D) {
        switch (method) {
            case RG_METHOD_PCG: f(D, IC<RG_METHOD_PCG>{}); return true;
            case RG_METHOD_PCG_PLAIN: f(D, IC<RG_METHOD_PCG_PLAIN>{}); return true;
            case RG_METHOD_BICGSTAB: f(D, IC<RG_METHOD_BICGSTAB>{}); return true;
            case RG_METHOD_MINRES: f(D, IC<RG_METHOD_MINRES>{}); return true;
            default: return false;
        }
    };
    return dim == 2 ? go(IC<2>{}) : go(IC<3>{});
}

}  // namespace

bool resident_fits(const rg_matrix* m, int method, int (&t)[3])
{
    const Geom& g = m->g;
    if (g.bs != 1 || g.N > (int64_t)kMaxTiles * kResThreads * 4) return false;
    bool fits = false;
    by_method(g.dim, method, [&](auto D, auto T) {
        fits = resident_tiles(g.dim, g.nn, kResThreads * res_rows<D.value, T.value>(),
                              kResThreads * res_cells<D.value, T.value>(), std::min(kMaxTiles, m->ctx->num_cu), t, 0.0);
    });
    return fits;
}

size_t resident_slot_bytes() { return sizeof(unsigned long long) * kSets * kMaxTiles * kMaxSums; }

namespace {

ResSystem res_system(const rg_matrix* m, const double* dinv, const int (&t)[3])
{
    const Geom& g = m->g;
    ResSystem s;
    s.val = m->val;
    s.dinv = dinv;
    s.ld = g.ld;
    s.n0 = (int)g.nn[0];
    s.n1 = (int)g.nn[1];
    s.n2 = g.dim == 3 ? (int)g.nn[2] : 1;
    s.tx = t[0];
    s.ty = t[1];
    s.tz = g.dim == 3 ? t[2] : 1;
    s.gx = (s.n0 + s.tx - 1) / s.tx;
    s.gy = (s.n1 + s.ty - 1) / s.ty;
    s.gz = (s.n2 + s.tz - 1) / s.tz;
    s.sym = m->symmetric;
    return s;
}

}  // namespace

ResEnd resident_solve(rg_matrix* m, int method, const int (&t)[3], int maxit, double tol, unsigned spins,
                      KrylovState* out)
{
    const Geom& g = m->g;
    rg_solver_work* w = m->work;
    hipStream_t st = m->ctx->stream;
    ResArgs a;
    a.sys = res_system(m, m->dinv, t);
    a.r = w->r;
    a.x = w->xw;
    a.pub0 = w->z;
    a.pub1 = w->z2;
    a.pub2 = w->s;
    a.slots = reinterpret_cast<unsigned long long*>(w->slots);
    a.st = w->st;
    a.maxit = maxit;
    a.tol = tol;
    a.spins = spins;
    const int tiles = a.sys.gx * a.sys.gy * a.sys.gz;
    const int cells = (a.sys.tx + 2) * (a.sys.ty + 2) * (g.dim == 3 ? a.sys.tz + 2 : 1);
    hipLaunchKernelGGL(k_res_empty, dim3(8), dim3(512), 0, st, a.slots, (int64_t)kSets * tiles * kMaxSums, w->st, 1);
    hipError_t err = hipErrorUnknown;
    by_method(g.dim, method, [&](auto D, auto T) {
        void* args[] = {&a};
        constexpr int rows = kResThreads * res_rows<D.value, T.value>();
        constexpr int vecs = T.value == RG_METHOD_BICGSTAB ? 2 : 1, own = T.value == RG_METHOD_PCG ? 2 : 1;
        static_assert(sizeof(double) * (vecs * kResThreads * res_cells<D.value, T.value>() + own * rows) +
                              sizeof(ResShared) <= 65536, "the tile outgrew the LDS");
        const unsigned lds = (unsigned)(sizeof(double) * (vecs * cells + own * rows));
        // all workgroups wait for one another: a cooperative launch starts
        // them together or not at all (one alone needs none)
        const void* kernel = reinterpret_cast<const void*>(k_resident<D.value, T.value>);
        err = tiles == 1 ? hipLaunchKernel(kernel, dim3(1), dim3(kResThreads), args, lds, st)
                         : hipLaunchCooperativeKernel(kernel, dim3(tiles), dim3(kResThreads), args, lds, st);
    });
    if (err != hipSuccess) {
        (void)hipGetLastError();
        return ResEnd::refused;
    }
    KrylovState* pin = reinterpret_cast<KrylovState*>(m->ctx->pinned);
    RG_HIP(hipMemcpyAsync(pin, w->st, sizeof(KrylovState), hipMemcpyDeviceToHost, st));
    RG_HIP(hipStreamSynchronize(st));
    *out = *pin;
    return out->done && !out->gave_up ? ResEnd::done : ResEnd::gave_up;
}

// --------------------------------------------------------------- batches

ResidentBatch::~ResidentBatch()
{
    if (mem) (void)hipFree(mem);
}

bool ResidentBatch::plan(const std::vector<rg_matrix*>& mats)
{
    if (state != RES_UNKNOWN) return res_on(state);
    state = RES_OFF;
    const rg_context* ctx = mats[0]->ctx;
    const int dim = mats[0]->g.dim, blocks = std::min(kMaxTiles, ctx->num_cu);
    const int rows = kResThreads * (dim == 2 ? kBatchRows2 : kBatchRows3), cap = rows + 3 * kResThreads;
    std::vector<double> time;
    int64_t sum = 0;
    tile.resize(3 * mats.size());
    for (size_t j = 0; j < mats.size(); ++j) {
        const Geom& g = mats[j]->g;
        int t[3];
        if (g.N > (int64_t)rows * blocks || !resident_tiles(dim, g.nn, rows, cap, blocks, t, 1.0)) return false;
        int G = 1;
        for (int d = 0; d < dim; ++d) G *= (int)((g.nn[d] + t[d] - 1) / t[d]);
        for (int d = 0; d < 3; ++d) tile[3 * j + d] = dim == 2 && d == 2 ? 1 : t[d];
        tiles.push_back(G);
        sum += G;
        const int64_t side = std::max(g.nn[0], std::max(g.nn[1], dim == 3 ? g.nn[2] : 1));
        time.push_back((double)side * (G > 1 ? 4.0 + 0.6 * std::log2((double)G) : 2.0));
    }
    grid = (int)std::min<int64_t>(blocks, sum);
    std::vector<int32_t> system, rank;
    resident_schedule(time, tiles, grid, first, system, rank);
    for (size_t k = 0; k < system.size(); ++k) {
        tasks.push_back(system[k]);
        tasks.push_back(rank[k]);
    }
    state = RES_FITS;
    return true;
}

ResEnd ResidentBatch::solve(const std::vector<rg_matrix*>& mats, const std::vector<int64_t>& off, const double* dinv,
                          const double* b, double* x, double* pub0, double* pub1, KrylovState* st, int maxit, double tol,
                          unsigned spins, std::vector<KrylovState>& out)
{
    const rg_context* ctx = mats[0]->ctx;
    hipStream_t s = ctx->stream;
    const int dim = mats[0]->g.dim;
    const size_t count = mats.size(), ntask = tasks.size() / 2;
    std::vector<int64_t> slot(count + 1, 0);
    for (size_t j = 0; j < count; ++j) slot[j + 1] = slot[j] + (int64_t)kSets * tiles[j] * kMaxSums;
    // systems, tasks, first, slots in one allocation (16-byte aligned parts)
    auto up = [](size_t n) { return (n + 15) / 16 * 16; };
    const size_t at_tasks = up(sizeof(ResBatchSystem) * count), at_first = at_tasks + up(sizeof(ResTask) * ntask),
                 at_slots = at_first + up(sizeof(int) * first.size()), bytes = at_slots + 8 * (size_t)slot[count];
    if (!mem) RG_HIP(hipMalloc(&mem, bytes));
    char* base = static_cast<char*>(mem);
    unsigned long long* slots = reinterpret_cast<unsigned long long*>(base + at_slots);
    std::vector<char> host(at_slots, 0);
    for (size_t j = 0; j < count; ++j) {
        const int t[3] = {tile[3 * j], tile[3 * j + 1], tile[3 * j + 2]};
        ResBatchSystem h;
        h.sys = res_system(mats[j], dinv + off[j], t);
        h.b = b + off[j];
        h.x = x + off[j];
        h.pub0 = pub0 + off[j];
        h.pub1 = pub1 + off[j];
        h.slots = slots + slot[j];
        std::memcpy(host.data() + sizeof(ResBatchSystem) * j, &h, sizeof(h));
    }
    static_assert(sizeof(ResTask) == 2 * sizeof(int32_t), "tasks are pairs");
    std::memcpy(host.data() + at_tasks, tasks.data(), sizeof(int32_t) * tasks.size());
    std::memcpy(host.data() + at_first, first.data(), sizeof(int) * first.size());
    RG_HIP(hipMemcpyAsync(mem, host.data(), host.size(), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_res_empty, dim3(64), dim3(512), 0, s, slots, slot[count], st, (int)count);
    ResBatchArgs a;
    a.systems = reinterpret_cast<const ResBatchSystem*>(base);
    a.tasks = reinterpret_cast<const ResTask*>(base + at_tasks);
    a.first = reinterpret_cast<const int*>(base + at_first);
    a.st = st;
    a.maxit = maxit;
    a.spins = spins;
    a.tol = tol;
    void* args[] = {&a};
    int cells = 0;
    for (size_t j = 0; j < count; ++j)
        cells = std::max(cells, (tile[3 * j] + 2) * (tile[3 * j + 1] + 2) * (dim == 3 ? tile[3 * j + 2] + 2 : 1));
    const int rows = kResThreads * (dim == 2 ? kBatchRows2 : kBatchRows3);
    static_assert(sizeof(double) * (2 * kBatchRows2 + 3) * kResThreads + sizeof(ResShared) <= 65536, "LDS");
    const unsigned lds = (unsigned)(sizeof(double) * (cells + rows));
    const void* kernel = dim == 2 ? reinterpret_cast<const void*>(k_resident_batch<2>)
                                  : reinterpret_cast<const void*>(k_resident_batch<3>);
    const hipError_t err = hipLaunchCooperativeKernel(kernel, dim3(grid), dim3(kResThreads), args, lds, s);
    if (err != hipSuccess) {
        (void)hipGetLastError();
        RG_HIP(hipStreamSynchronize(s));
        return ResEnd::refused;
    }
    out.resize(count);
    RG_HIP(hipMemcpyAsync(out.data(), st, sizeof(KrylovState) * count, hipMemcpyDeviceToHost, s));
    RG_HIP(hipStreamSynchronize(s));
    for (const KrylovState& k : out)
        if (!k.done || k.gave_up) return ResEnd::gave_up;
    return ResEnd::done;
}

}  // namespace rg
