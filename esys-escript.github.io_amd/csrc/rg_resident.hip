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

#include "rg_device.h"
#include "rg_resident.h"
#include "rg_stencil.h"

namespace rg {

namespace {

constexpr int kResThreads = 512;   // two waves per SIMD, 256 registers each
constexpr int kResWaves = kResThreads / 64;
constexpr int kMaxSums = 4;        // sums of one reduction
constexpr int kSets = 4;           // sets of slots
constexpr int kMaxTiles = 256;     // one per CU
constexpr unsigned long long kEmpty = 0xFFF8DEADBEEF0001ull;   // a NaN no sum is stored as

struct ResArgs {
    const double* val;
    const double* dinv;
    const double* r;
    double* x;
    double* pub0;        // surface values by node
    double* pub1;
    double* pub2;
    unsigned long long* slots;
    KrylovState* st;
    int64_t ld;
    int N, n0, n1, n2;
    int tx, ty, tz;      // tile sides
    int gx, gy;          // tiles per axis
    int sym, maxit;
    unsigned spins;      // polls of a slot before a workgroup gives up
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

// Totals of v over all workgroups (valid in all threads, the same bits in
// all workgroups); false once a workgroup has waited too long, whereupon
// every workgroup ends.
template <int NV>
__device__ __forceinline__ bool reduce_all(ResShared& sh, const ResArgs& a, unsigned& epoch, double (&v)[NV])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, G = gridDim.x;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const double s = wave_total(v[k]);
        if (lane == 0) sh.red[k][w] = s;
    }
    __builtin_amdgcn_s_waitcnt(0);   // this wave's surface values and emptied slots have arrived
    __syncthreads();
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
            unsigned long long* cur = a.slots + (size_t)(epoch & (kSets - 1)) * kMaxTiles * kMaxSums;
            unsigned long long* nxt = a.slots + (size_t)((epoch + 2) & (kSets - 1)) * kMaxTiles * kMaxSums;
#pragma unroll
            for (int k = 0; k < NV; ++k)
                if (lane == k)
                    put(cur + blockIdx.x * kMaxSums + k,
                        s[k] == s[k] ? (unsigned long long)__double_as_longlong(s[k]) : 0x7FF8000000000000ull);
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
            if (lane < kMaxSums) put(nxt + blockIdx.x * kMaxSums + lane, kEmpty);
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

// Rows per thread: as many as leave the stencil rows and the method's
// vectors in 256 registers.
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

// The recurrences are those of the launch sequences (stage_apply and the
// update kernels of the solver): PASO's residual-smoothed PCG, the textbook
// PCG, BiCGStab and MINRES with one Jacobi sweep, and the same stopping
// tests in the same order.
template <int DIM, int METHOD>
__global__ __launch_bounds__(kResThreads) void k_resident(ResArgs a)
{
    constexpr int NS = StencilShape<DIM>::NS;
    constexpr int CEN = StencilShape<DIM>::CENTER;
    constexpr int M = res_rows<DIM, METHOD>();
    constexpr int KH = res_cells<DIM, METHOD>();
    constexpr bool BICG = METHOD == RG_METHOD_BICGSTAB;
    __shared__ ResShared sh;
    extern __shared__ double lds[];
    const int tid = threadIdx.x, G = gridDim.x;
    const int px = a.tx + 2, py = a.ty + 2, pz = DIM == 3 ? a.tz + 2 : 1;
    const int cells = px * py * pz;
    double* P = lds;             // the vector the operator is applied to
    double* S = lds + cells;     // BiCGStab: the second one
    double* X = lds + (BICG ? 2 : 1) * cells + tid;   // the iterate of this thread's rows
    double* X2 = X + M * kResThreads;                 // PASO: the unsmoothed one
    const int bx = blockIdx.x % a.gx, by = (blockIdx.x / a.gx) % a.gy, bz = blockIdx.x / (a.gx * a.gy);
    const int x0 = bx * a.tx, y0 = by * a.ty, z0 = bz * a.tz;
    const int s1 = a.n0, s2 = a.n0 * a.n1;

    // halo cells of this thread: node of padded cell tid + k * threads, -1
    // for the tile's own cells and outside the grid
    int halo[KH];
#pragma unroll
    for (int k = 0; k < KH; ++k) {
        const int c = tid + k * kResThreads;
        halo[k] = -1;
        if (c < cells) {
            const int cx = c % px, cy = (c / px) % py, cz = DIM == 3 ? c / (px * py) : 1;
            const int gx = x0 + cx - 1, gy = y0 + cy - 1, gz = DIM == 3 ? z0 + cz - 1 : 0;
            const bool own = cx >= 1 && cx <= a.tx && cy >= 1 && cy <= a.ty && (DIM == 2 || (cz >= 1 && cz <= a.tz));
            const bool in = gx >= 0 && gx < a.n0 && gy >= 0 && gy < a.n1 && gz >= 0 && gz < a.n2;
            if (!own && in) halo[k] = gx + s1 * gy + s2 * gz;
            P[c] = 0.0;
            if constexpr (BICG) S[c] = 0.0;
        }
    }
    // own rows: node, padded cell, surface flag; a row outside the tile's
    // part of the grid has node -1, a zero stencil and reads cell 0
    int node[M], cell[M];
    bool surf[M];
    double A[M][NS], di[M], r[M];
    const int tile = a.tx * a.ty * (DIM == 3 ? a.tz : 1);
#pragma unroll
    for (int j = 0; j < M; ++j) {
        const int l = tid + j * kResThreads;
        const int lx = l % a.tx, ly = (l / a.tx) % a.ty, lz = DIM == 3 ? l / (a.tx * a.ty) : 0;
        const bool in = l < tile && x0 + lx < a.n0 && y0 + ly < a.n1 && (DIM == 2 || z0 + lz < a.n2);
        node[j] = in ? (x0 + lx) + s1 * (y0 + ly) + s2 * (DIM == 3 ? z0 + lz : 0) : -1;
        // (an interior cell of the padded tile, so that the stencil's reach stays inside it)
        cell[j] = in ? (lx + 1) + px * ((ly + 1) + (DIM == 3 ? py * (lz + 1) : 0)) : 1 + px * (1 + (DIM == 3 ? py : 0));
        surf[j] = in && G > 1 && (lx == 0 || lx == a.tx - 1 || ly == 0 || ly == a.ty - 1 ||
                                  (DIM == 3 && (lz == 0 || lz == a.tz - 1)));
        const int i = in ? node[j] : 0;
        di[j] = in ? a.dinv[i] : 0.0;
        r[j] = in ? a.r[i] : 0.0;
        X[j * kResThreads] = in ? a.x[i] : 0.0;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            int dx, dy, dz;
            slot_delta<DIM>(s, dx, dy, dz);
            double v;
            if (!a.sym) {
                v = a.val[(int64_t)s * a.ld + i];
            } else if (s >= CEN) {
                v = a.val[(int64_t)(s - CEN) * a.ld + i];
            } else {
                const int jn = i + dx + dy * s1 + dz * s2;
                v = jn >= 0 ? a.val[(int64_t)(CEN - s) * a.ld + jn] : 0.0;
            }
            A[j][s] = in ? v : 0.0;
        }
    }
    // Indices are made opaque at each use: kept over the iterations, the
    // addresses formed from them took some 60 registers.
    auto opaque = [](int i) {
        asm volatile("" : "+v"(i));
        return i;
    };
    auto apply = [&](const double* V, int j) {
        double acc = 0.0;
        const double* c = V + opaque(cell[j]);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            int dx, dy, dz;
            slot_delta<DIM>(s, dx, dy, dz);
            acc = fma(A[j][s], c[dx + px * (dy + py * dz)], acc);
        }
        __builtin_amdgcn_sched_barrier(0);   // one row's loads in flight at a time: registers
        return acc;
    };
    auto publish = [&](double* pub, int j, double v) {
        if (surf[j]) put(pub + opaque(node[j]), v);
    };
    auto own = [&](double* V, int j, double v) {
        if (node[j] >= 0) V[cell[j]] = v;
    };

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
                publish(a.pub0, j, z);
                t[0] = fma(z, r[j], t[0]);
                t[1] = fma(r[j], r[j], t[1]);
                if constexpr (PASO) {
                    rs[j] = r[j];
                    X2[j * kResThreads] = X[j * kResThreads];
                }
            }
            ok = reduce_all<2>(sh, a, epoch, t);
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
            for (int k = 0; k < KH; ++k) zh[k] = halo[k] >= 0 ? get(a.pub0 + opaque(halo[k])) : 0.0;
#pragma unroll
            for (int j = 0; j < M; ++j) own(P, j, fma(beta, P[cell[j]], di[j] * r[j]));
#pragma unroll
            for (int k = 0; k < KH; ++k)
                if (halo[k] >= 0) P[tid + k * kResThreads] = fma(beta, P[tid + k * kResThreads], zh[k]);
            __syncthreads();
            double q[M], d[1] = {0.0};
#pragma unroll
            for (int j = 0; j < M; ++j) {
                q[j] = apply(P, j);
                d[0] = fma(q[j], P[cell[j]], d[0]);
            }
            ok = reduce_all<1>(sh, a, epoch, d);
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
                    publish(a.pub0, j, z);
                    t[0] = fma(z, r[j], t[0]);
                    t[1] = fma(r[j], r[j], t[1]);
                }
#pragma unroll
                for (int j = 0; j < M; ++j)
                    X[j * kResThreads] = fma(alpha, P[cell[j]], X[j * kResThreads]);
                ok = reduce_all<2>(sh, a, epoch, t);
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
                    publish(a.pub0, j, z);
                    const double e = r[j] - rs[j];
                    t[0] = fma(e, e, t[0]);
                    t[1] = fma(e, rs[j], t[1]);
                    t[2] = fma(rs[j], rs[j], t[2]);
                    t[3] = fma(z, r[j], t[3]);
                    X2[j * kResThreads] = fma(alpha, P[cell[j]], X2[j * kResThreads]);
                }
                ok = reduce_all<4>(sh, a, epoch, t);
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
                    ok = reduce_all<1>(sh, a, epoch, nn);
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
                publish(a.pub0, j, z);
                t[0] = fma(r[j], z, t[0]);
                t[1] = fma(r[j], r[j], t[1]);
            }
            ok = reduce_all<2>(sh, a, epoch, t);
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
            for (int k = 0; k < KH; ++k) zh[k] = halo[k] >= 0 ? get(a.pub0 + opaque(halo[k])) : 0.0;
#pragma unroll
            for (int j = 0; j < M; ++j) own(P, j, ig * (di[j] * r[j]));
#pragma unroll
            for (int k = 0; k < KH; ++k)
                if (halo[k] >= 0) P[tid + k * kResThreads] = ig * zh[k];
            __syncthreads();
            double q[M], d[1] = {0.0};
#pragma unroll
            for (int j = 0; j < M; ++j) {
                q[j] = apply(P, j);
                d[0] = fma(q[j], P[cell[j]], d[0]);
            }
            ok = reduce_all<1>(sh, a, epoch, d);
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
                publish(a.pub0, j, z);
                t[0] = fma(v, z, t[0]);
            }
            ok = reduce_all<1>(sh, a, epoch, t);
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
                publish(a.pub0, j, di[j] * r[j]);
                publish(a.pub1, j, 0.0);
                t[0] = fma(rt[j], r[j], t[0]);
            }
            ok = reduce_all<1>(sh, a, epoch, t);
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
                h0[k] = halo[k] >= 0 ? get(a.pub0 + opaque(halo[k])) : 0.0;
                h1[k] = halo[k] >= 0 ? get(a.pub1 + opaque(halo[k])) : 0.0;
            }
#pragma unroll
            for (int j = 0; j < M; ++j) {
                p[j] = iter > 1 ? r[j] + beta * (p[j] - omega * v[j]) : r[j];
                own(P, j, di[j] * p[j]);
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
                v[j] = apply(P, j);
                publish(a.pub2, j, di[j] * v[j]);
                d[0] = fma(rt[j], v[j], d[0]);
            }
            ok = reduce_all<1>(sh, a, epoch, d);
            if (!ok) break;
            if (fabs(d[0]) <= 0.0) {
                status = KS_BREAKDOWN;
                break;
            }
            alpha = tau / d[0];
#pragma unroll
            for (int k = 0; k < KH; ++k) h0[k] = halo[k] >= 0 ? get(a.pub2 + opaque(halo[k])) : 0.0;
            double t[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int j = 0; j < M; ++j) {
                r[j] = fma(-alpha, v[j], r[j]);
                own(S, j, di[j] * r[j]);
                t[2] = fma(r[j], r[j], t[2]);
            }
#pragma unroll
            for (int k = 0; k < KH; ++k)
                if (halo[k] >= 0) S[tid + k * kResThreads] = fma(-alpha, h0[k], S[tid + k * kResThreads]);
            __syncthreads();
            double tv[M];
#pragma unroll
            for (int j = 0; j < M; ++j) {
                tv[j] = apply(S, j);
                t[0] = fma(tv[j], r[j], t[0]);
                t[1] = fma(tv[j], tv[j], t[1]);
            }
            ok = reduce_all<3>(sh, a, epoch, t);
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
                publish(a.pub0, j, di[j] * r[j]);
                publish(a.pub1, j, di[j] * (p[j] - omega * v[j]));
                e[0] = fma(r[j], r[j], e[0]);
                e[1] = fma(rt[j], r[j], e[1]);
            }
            ok = reduce_all<2>(sh, a, epoch, e);
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
    if (ok && blockIdx.x == 0 && tid == 0) {
        a.st->status = status;
        a.st->num_iter = iter;
        a.st->norm = norm;
        a.st->done = 1;
    }
}

__global__ void k_res_empty(unsigned long long* slots, KrylovState* st)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < kSets * kMaxTiles * kMaxSums; i += gridDim.x * blockDim.x)
        slots[i] = kEmpty;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->done = 0;
        st->status = KS_RUNNING;
        st->num_iter = 0;
        st->norm = 0.0;
        st->gave_up = 0;
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

// Tile sides for a grid of n nodes per axis: at most `rows` nodes and
// `cells` padded cells per tile and `tiles` tiles.  Among the shapes that
// fit, the one with the least estimated time per iteration: a reduction over
// G workgroups measured 1.6 / 2.3 / 2.7 / 3.2 / 3.7 / 4.0 us for G = 1 / 8 /
// 32 / 64 / 128 / 256, the stencil about 0.4 us (3-D) or 0.15 us (2-D) per
// 512 rows, a halo of 1024 cells 1.5 us.
bool resident_tiles(int dim, const int64_t* nn, int rows, int cells, int tiles, int (&t)[3])
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
                const double cost = (G > 1 ? 2.0 * (1.4 + 0.3 * std::log2((double)G)) + 1.0 + (pad - vol) / 1024.0 : 1.0) +
                                    (dim == 3 ? 0.4 : 0.15) * (double)((vol + 511) / 512);
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

bool resident_fits(const rg_matrix* m, int method, int (&t)[3])
{
    const Geom& g = m->g;
    if (g.bs != 1 || g.N > (int64_t)kMaxTiles * kResThreads * 4) return false;
    bool fits = false;
    by_method(g.dim, method, [&](auto D, auto T) {
        fits = resident_tiles(g.dim, g.nn, kResThreads * res_rows<D.value, T.value>(),
                              kResThreads * res_cells<D.value, T.value>(), std::min(kMaxTiles, m->ctx->num_cu), t);
    });
    return fits;
}

size_t resident_slot_bytes() { return sizeof(unsigned long long) * kSets * kMaxTiles * kMaxSums; }

bool resident_solve(rg_matrix* m, int method, const int (&t)[3], int maxit, double tol, unsigned spins, KrylovState* out)
{
    const Geom& g = m->g;
    rg_solver_work* w = m->work;
    hipStream_t st = m->ctx->stream;
    ResArgs a;
    a.val = m->val;
    a.dinv = m->dinv;
    a.r = w->r;
    a.x = w->xw;
    a.pub0 = w->z;
    a.pub1 = w->z2;
    a.pub2 = w->s;
    a.slots = reinterpret_cast<unsigned long long*>(w->slots);
    a.st = w->st;
    a.ld = g.ld;
    a.N = (int)g.N;
    a.n0 = (int)g.nn[0];
    a.n1 = (int)g.nn[1];
    a.n2 = g.dim == 3 ? (int)g.nn[2] : 1;
    a.tx = t[0];
    a.ty = t[1];
    a.tz = g.dim == 3 ? t[2] : 1;
    a.gx = (a.n0 + a.tx - 1) / a.tx;
    a.gy = (a.n1 + a.ty - 1) / a.ty;
    const int gz = (a.n2 + a.tz - 1) / a.tz;
    a.sym = m->symmetric;
    a.maxit = maxit;
    a.tol = tol;
    a.spins = spins;
    const int cells = (a.tx + 2) * (a.ty + 2) * (g.dim == 3 ? a.tz + 2 : 1);
    hipLaunchKernelGGL(k_res_empty, dim3(8), dim3(512), 0, st, a.slots, w->st);
    hipError_t err = hipErrorUnknown;
    by_method(g.dim, method, [&](auto D, auto T) {
        void* args[] = {&a};
        constexpr int rows = kResThreads * res_rows<D.value, T.value>();
        constexpr int vecs = T.value == RG_METHOD_BICGSTAB ? 2 : 1, own = T.value == RG_METHOD_PCG ? 2 : 1;
        static_assert(sizeof(double) * (vecs * kResThreads * res_cells<D.value, T.value>() + own * rows) +
                              sizeof(ResShared) <= 65536, "the tile outgrew the LDS");
        const unsigned lds = (unsigned)(sizeof(double) * (vecs * cells + own * rows));
        // all workgroups wait for one another: a cooperative launch starts
        // them together or not at all
        err = hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_resident<D.value, T.value>),
                                         dim3(a.gx * a.gy * gz), dim3(kResThreads), args, lds, st);
    });
    if (err != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    KrylovState* pin = reinterpret_cast<KrylovState*>(m->ctx->pinned);
    RG_HIP(hipMemcpyAsync(pin, w->st, sizeof(KrylovState), hipMemcpyDeviceToHost, st));
    RG_HIP(hipStreamSynchronize(st));
    *out = *pin;
    return out->done && !out->gave_up;
}

}  // namespace rg
