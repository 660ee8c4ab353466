// Matrix kernels of libripley_hip: value initialisation, element-block
// insertion, colour-free gather assembly, stencil SpMV, Dirichlet
// nullification and the PASO CSR export.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>

#include "rg_device.h"
#include "rg_dispatch.h"
#include "rg_stencil.h"

namespace rg {

// ------------------------------------------------------------- set values
// paso::SystemMatrix::setValues (paso/src/SystemMatrix.h:273-279): every
// entry of the PASO pattern := value.  Stencil slots whose neighbour lies
// outside the grid are not in the pattern and are set to zero.
template <int DIM, int BS, bool SYM>
__global__ __launch_bounds__(kBlock) void k_set_values(double* __restrict__ val, int64_t ld, int64_t N,
                                                       int64_t n0, int64_t n1, int64_t n2,
                                                       double value)
{
    constexpr int NST = stored_slots<DIM, SYM>();
    constexpr int FIRST = SYM ? StencilShape<DIM>::CENTER : 0;
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= N) return;
    const int64_t x = i % n0, y = (i / n0) % n1, z = i / (n0 * n1);
#pragma unroll
    for (int t = 0; t < NST; ++t) {
        const double v = slot_in_grid<DIM>(FIRST + t, x, y, z, n0, n1, n2) ? value : 0.0;
#pragma unroll
        for (int e = 0; e < BS * BS; ++e) val[(int64_t)(t * BS * BS + e) * ld + i] = v;
    }
}

void launch_set_values(rg_matrix* m, double value)
{
    const Geom& g = m->g;
    const int grid = (int)((g.N + kBlock - 1) / kBlock);
    dispatch(g, m->symmetric, [&](auto D, auto B, auto S) {
        hipLaunchKernelGGL((k_set_values<D.value, B.value, S.value>), dim3(grid), dim3(kBlock), 0,
                           m->ctx->stream, m->val, g.ld, g.N, g.nn[0], g.nn[1], g.nn[2], value);
    });
    RG_HIP(hipGetLastError());
    m->val_zero = (value == 0.0);
}

// -------------------------------------------------- element block insertion
// ripley::SystemMatrix::add (ripley/src/RipleySystemMatrix.cu:111-155), the
// stencil-matrix counterpart of addToPasoMatrix
// (ripley/src/RipleyDomain.cpp:1488-1517): the pair (a, b) of local element
// nodes lands in the slot given by their local positions; with symmetric
// storage only pairs with b >= a are added.
//
// One launch per element colour: the colour of an element is the parity of
// the grid coordinates of its local node 0 (2^DIM colours), so two distinct
// grid cells of one colour share no node -- the slab colouring that makes
// the reference's assembler loops race-free (DefaultAssembler3D.cpp:243-245),
// taken in all axes.  Inside a launch every thread owns one (element, a, b,
// k, m) target.  For distinct grid cells each matrix entry then receives at
// most one contribution per launch and the sums are formed in colour order,
// the same on every run.  The adds are atomic, so inputs whose "elements"
// share nodes within a colour (repeated elements, node lists that are not
// grid cells) stay race-free; only their summation order is then open.
template <int DIM, int BS, bool SYM>
__global__ __launch_bounds__(kBlock) void k_add_elements(double* __restrict__ val, int64_t ld, int64_t n0,
                                                         int64_t n1, int64_t num_el,
                                                         const int32_t* __restrict__ nodes,
                                                         const double* __restrict__ em, int colour)
{
    constexpr int NN = 1 << DIM;
    constexpr int C = StencilShape<DIM>::CENTER;
    constexpr int NT = NN * NN * BS * BS;
    const int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (t >= num_el * NT) return;
    const int64_t e = t / NT;
    const int j = (int)(t - e * NT);
    const int64_t base = nodes[e * NN];
    const int64_t bx = base % n0, by = (base / n0) % n1, bz = base / (n0 * n1);
    const int c = (int)((bx & 1) | ((by & 1) << 1) | (DIM == 3 ? (bz & 1) << 2 : 0));
    if (c != colour) return;
    const int k = j % BS, mm = (j / BS) % BS, a = (j / (BS * BS)) % NN, b = j / (BS * BS * NN);
    if (SYM && b < a) return;
    const int s = ((b & 1) - (a & 1) + 1) + 3 * (((b >> 1) & 1) - ((a >> 1) & 1) + 1) +
                  (DIM == 3 ? 9 * (((b >> 2) & 1) - ((a >> 2) & 1) + 1) : 0);
    const int st = SYM ? s - C : s;
    const int64_t row = nodes[e * NN + a];
    atomicAdd(&val[(int64_t)(st * BS * BS + k + BS * mm) * ld + row], em[t]);
}

void launch_add_element_blocks(rg_matrix* m, int64_t ne, int npe, const int32_t* d_nodes,
                               const double* d_em)
{
    const Geom& g = m->g;
    RG_CHECK(npe == (1 << g.dim), RG_VALUE_ERROR,
             "add_element_blocks: nodes_per_element must be 4 (2-D) or 8 (3-D)");
    if (ne == 0) return;
    const int64_t targets = ne * npe * npe * g.bs * g.bs;
    const int64_t grid = (targets + kBlock - 1) / kBlock;
    RG_CHECK(grid < ((int64_t)1 << 31), RG_VALUE_ERROR, "add_element_blocks: too many elements in one call");
    dispatch(g, m->symmetric, [&](auto D, auto B, auto S) {
        for (int c = 0; c < npe; ++c)
            hipLaunchKernelGGL((k_add_elements<D.value, B.value, S.value>), dim3((unsigned)grid), dim3(kBlock), 0,
                               m->ctx->stream, m->val, g.ld, g.nn[0], g.nn[1], ne, d_nodes, d_em, c);
    });
    RG_HIP(hipGetLastError());
    m->val_zero = false;
}

// ---------------------------------------------------- allocation-free scratch
// Device memory of the entry points that allocate nothing
// (rg_matrix_add_element_blocks_noalloc): one array per device, held until
// the process ends.  Host code must not pass the array's name to a kernel
// (it is a host-side stand-in); it uses the device address that
// scratch_address() looks up once per device with that device current.
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

void* scratch_address()
{
    constexpr int kMaxDevices = 64;
    static std::mutex mu;
    static void* addr[kMaxDevices] = {};
    int dev = 0;
    RG_HIP(hipGetDevice(&dev));
    RG_CHECK(dev >= 0 && dev < kMaxDevices, RG_DEVICE_ERROR, "scratch: device id out of range");
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        void* p = nullptr;
        RG_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        RG_CHECK(p != nullptr, RG_DEVICE_ERROR, "hipGetSymbolAddress(scratch) returned NULL");
        addr[dev] = p;
    }
    return addr[dev];
}

// ---------------------------------------------------------------- assembly
struct CoefDev {
    const double* p;
    int mode;
    int stride;
    int iso;
};
struct AsmArgs {
    CoefDev A, B, C, D, X, Y;
    int64_t n0, n1, n2;     // nodes per axis
    int ne0, ne1, ne2;      // elements per axis
    double h0, h1, h2;
};

__device__ __forceinline__ const double* coef_pt(const CoefDev& c, int64_t e, int q, int dps)
{
    const double* p = c.p + (int64_t)c.stride * e;
    return (c.mode == RG_COEF_EXPANDED) ? p + q * dps : p;
}

// Nodes whose (k, m) pairs one wave holds.
template <int NB>
__host__ __device__ constexpr int asm_nodes_per_wave()
{
    return 64 / (NB * NB);
}

// Colour-free gather assembly.  One thread per (node i, equation k,
// component m): it visits the 2^DIM elements around node i, forms row a (the
// node's local index) of each element matrix and adds entry (a, b) to the
// stencil slot of local node b:
//   EM_S[k,m,a,b] = int A[k,i,m,j] dN_a/dx_i dN_b/dx_j + B[k,i,m] N_b dN_a/dx_i
//                     + C[k,m,j] N_a dN_b/dx_j + D[k,m] N_a N_b
//   EM_F[k,a]     = int X[k,i] dN_a/dx_i + Y[k] N_a
// -- the weak form that DefaultAssembler3D::assemblePDESingle/System
// integrate with the 2-point Gauss rule (points (1-+1/sqrt3)/2, x fastest;
// ripley/src/DefaultAssembler3D.cpp:153-2229, :3631-5745) and, for reduced,
// the one-point rule of assemblePDE*Reduced (:2891-3270).  Each matrix entry
// and rhs entry is written by exactly one thread: no atomics.
//
// Coefficients with one point per element (k_assemble_const) are integrated
// in closed form (the 2-point rule is exact for these products): along an axis
// int N N = 1/3 or 1/6 for equal / different local coordinates, int N' N =
// +-1/2, int N' N' = +-1 in units of h, so an entry takes one multiply-add
// per coefficient component instead of one Gauss sum.  The one-point rule
// differs in int N N = 1/4 only (ONE): as a Gauss sum its single point paid
// the staging for nothing, A, D, X, Y on Brick 70x60x50 113 us, closed form
// 66 us (the whole call).  Coefficients on quadrature points (k_assemble_gauss) take the
// Gauss sum, the point loop outermost so that the shape functions of a point
// serve all elements.  Both in one kernel took 256 registers (one wave per
// SIMD); a PDE with both kinds runs a launch of each.
//
// Bound: the coefficient reads.  A data point of a system is NB^2 DIM^2 (A)
// contiguous doubles of which thread (k, m) needs every NB-th, so the lanes
// of a wave are the NB^2 pairs (k, m) of 64 / NB^2 neighbouring nodes: one
// load instruction then covers whole runs of a data point, and the block's
// four waves take 2 x 2 neighbouring node lines (3-D; four lines in 2-D),
// which share their elements through L1.  With one (k, m) per blockIdx.y and
// lanes along x, each load touched 64 lines: Brick 48x47x49, 3 equations,
// A per element and the rest on quadrature points 10.48 ms -> 0.17 + 0.77 ms (bytes alone 0.24 ms);
// Brick 96^3 elasticity (A per element, symmetric storage) 37.6 -> 0.92 ms (bytes alone 0.30 ms).
//
// The block's nodes are those of an AsmTile: the wide one (64 / NB^2 x 2 x 2),
// whose sides the compiler knows, or the one given (TILE, asm_tile).
template <int DIM, int NB, bool TILE>
struct AsmNode {
    int k, m;            // equation and component of the thread
    int64_t x, y, z, i;  // its node
    bool valid;
    int64_t e0;          // element at (x - 1, y - 1, z - 1)
    unsigned in;         // bit t: element t = (ex, ey, ez) at node index - 1 + t is in the grid
    int corner;          // element (x - 1, y - 1, z - 1) among those of the block
    __device__ __forceinline__ AsmNode(const AsmArgs& a, const AsmTile& t)
    {
        constexpr int PAIRS = NB * NB, NPW = asm_nodes_per_wave<NB>();
        const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
        const int km = lane % PAIRS;
        k = km % NB;
        m = km / NB;
        const int wx = TILE ? t.wx : NPW, wy = TILE ? t.wy : asm_wide_y(DIM), wz = TILE ? t.wz : asm_wide_z(DIM);
        int lx = lane / PAIRS, ly = DIM == 3 ? wv & 1 : wv, lz = DIM == 3 ? wv >> 1 : 0;
        bool in_tile = lane < PAIRS * NPW;
        if (TILE) {
            const int l = wv * NPW + lx;         // node of the tile, x fastest
            in_tile = in_tile && l < wx * wy * wz;
            lx = l % wx;
            ly = (l / wx) % wy;
            lz = DIM == 3 ? l / (wx * wy) : 0;
        }
        corner = in_tile ? lx + (wx + 1) * (ly + (wy + 1) * lz) : 0;
        const int64_t bx = blockIdx.x % t.gx, by = (blockIdx.x / t.gx) % t.gy, bz = blockIdx.x / (t.gx * t.gy);
        x = bx * wx + lx;
        y = by * wy + ly;
        z = DIM == 3 ? bz * wz + lz : 0;
        valid = in_tile && x < a.n0 && y < a.n1 && (DIM == 2 || z < a.n2);
        i = x + a.n0 * (y + (DIM == 3 ? a.n1 * z : 0));
        e0 = (x - 1) + (int64_t)a.ne0 * ((y - 1) + (DIM == 3 ? (int64_t)a.ne1 * (z - 1) : 0));
        in = 0;
#pragma unroll
        for (int t = 0; t < (1 << DIM); ++t) {
            const int64_t k0 = x - 1 + (t & 1), k1 = y - 1 + ((t >> 1) & 1), k2 = (DIM == 3) ? z - 1 + (t >> 2) : 0;
            if (k0 >= 0 && k0 < a.ne0 && k1 >= 0 && k1 < a.ne1 && (DIM == 2 || (k2 >= 0 && k2 < a.ne2))) in |= 1u << t;
        }
    }
    __device__ __forceinline__ int64_t element(const AsmArgs& a, int t) const
    {
        return e0 + (t & 1) + (int64_t)a.ne0 * (((t >> 1) & 1) + (DIM == 3 ? (int64_t)a.ne1 * (t >> 2) : 0));
    }
};

// Stencil slot of local node b of element t, seen from the node.
template <int DIM>
__host__ __device__ constexpr int asm_slot(int t, int b)
{
    return ((t & 1) + (b & 1)) + 3 * (((t >> 1) & 1) + ((b >> 1) & 1)) + (DIM == 3 ? 9 * ((t >> 2) + (b >> 2)) : 0);
}

template <int DIM, int NB, bool SYM, bool TILE>
__device__ __forceinline__ void asm_store(const AsmNode<DIM, NB, TILE>& nd, const double (&acc)[StencilShape<DIM>::NS],
                                          double* __restrict__ val, int64_t ld, bool zero)
{
    constexpr int FIRST = SYM ? StencilShape<DIM>::CENTER : 0;
#pragma unroll
    for (int t = 0; t < stored_slots<DIM, SYM>(); ++t) {
        double* p = &val[(int64_t)(t * NB * NB + nd.k + NB * nd.m) * ld + nd.i];
        if (zero) *p = acc[FIRST + t];
        else *p += acc[FIRST + t];
    }
}

template <int DIM, int NB, bool SYM, bool ONE, bool TILE>
__global__ __launch_bounds__(kBlock) void k_assemble_const(AsmArgs a, AsmTile tile, double* __restrict__ val,
                                                           int64_t ld, bool zero, double* __restrict__ rhs)
{
    constexpr int NS = StencilShape<DIM>::NS;
    constexpr int NNODE = 1 << DIM;
    const AsmNode<DIM, NB, TILE> nd(a, tile);
    if (!nd.valid) return;
    const int k = nd.k, m = nd.m;
    const double ih[3] = {1.0 / a.h0, 1.0 / a.h1, 1.0 / a.h2};
    double vol = a.h0 * a.h1;
    if (DIM == 3) vol *= a.h2;
    const bool doS = (a.A.mode | a.B.mode | a.C.mode | a.D.mode) != 0;
    const bool doF = rhs != nullptr && m == 0 && (a.X.mode | a.Y.mode) != 0;
    double acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s] = 0.0;
    double f = 0.0;
#pragma unroll
    for (int t = 0; t < NNODE; ++t) {
        if (nd.in & (1u << t)) {
            const int64_t e = nd.element(a, t);
            double A[DIM][DIM], B[DIM], C[DIM], D = 0.0;
#pragma unroll
            for (int p = 0; p < DIM; ++p) {
                B[p] = C[p] = 0.0;
#pragma unroll
                for (int j = 0; j < DIM; ++j) A[p][j] = 0.0;
            }
            if (a.A.mode) {
                const double* P = a.A.p + (int64_t)a.A.stride * e;
                if (a.A.iso) {
#pragma unroll
                    for (int p = 0; p < DIM; ++p) A[p][p] = P[0] * (vol * ih[p] * ih[p]);
                } else {
#pragma unroll
                    for (int j = 0; j < DIM; ++j)
#pragma unroll
                        for (int p = 0; p < DIM; ++p)
                            A[p][j] = P[k + NB * (p + DIM * (m + NB * j))] * (vol * ih[p] * ih[j]);
                }
            }
            if (a.B.mode) {
                const double* P = a.B.p + (int64_t)a.B.stride * e;
#pragma unroll
                for (int p = 0; p < DIM; ++p) B[p] = P[k + NB * (p + DIM * m)] * (vol * ih[p]);
            }
            if (a.C.mode) {
                const double* P = a.C.p + (int64_t)a.C.stride * e;
#pragma unroll
                for (int p = 0; p < DIM; ++p) C[p] = P[k + NB * (m + NB * p)] * (vol * ih[p]);
            }
            if (a.D.mode) D = (a.D.p + (int64_t)a.D.stride * e)[k + NB * m] * vol;
#pragma unroll
            for (int b = 0; b < NNODE; ++b) {
                const int s = asm_slot<DIM>(t, b);
                if (SYM && s < StencilShape<DIM>::CENTER) continue;
                // signs of dN_a, dN_b and int N_a N_b / h along each axis
                double sa[DIM], sb[DIM], mass[DIM];
#pragma unroll
                for (int p = 0; p < DIM; ++p) {
                    const int ab = 1 - ((t >> p) & 1), bb = (b >> p) & 1;
                    sa[p] = ab ? 1.0 : -1.0;
                    sb[p] = bb ? 1.0 : -1.0;
                    mass[p] = ONE ? 0.25 : ab == bb ? 1.0 / 3.0 : 1.0 / 6.0;
                }
                double full = 1.0, r = acc[s];
#pragma unroll
                for (int p = 0; p < DIM; ++p) full *= mass[p];
#pragma unroll
                for (int p = 0; p < DIM; ++p)
#pragma unroll
                    for (int j = 0; j < DIM; ++j) {
                        double c = (p == j) ? sa[p] * sb[p] : 0.25 * sa[p] * sb[j];
#pragma unroll
                        for (int o = 0; o < DIM; ++o)
                            if (o != p && o != j) c *= mass[o];
                        r = fma(A[p][j], c, r);
                    }
                if (a.B.mode | a.C.mode) {
#pragma unroll
                    for (int p = 0; p < DIM; ++p) {
                        double c = 0.5;
#pragma unroll
                        for (int o = 0; o < DIM; ++o)
                            if (o != p) c *= mass[o];
                        r = fma(B[p], c * sa[p], r);
                        r = fma(C[p], c * sb[p], r);
                    }
                }
                acc[s] = fma(D, full, r);
            }
            if (doF) {
                if (a.X.mode) {
                    const double* P = a.X.p + (int64_t)a.X.stride * e;
#pragma unroll
                    for (int p = 0; p < DIM; ++p) {
                        const double c = ((t >> p) & 1) ? -2.0 / NNODE : 2.0 / NNODE;
                        f = fma(P[k + NB * p], c * (vol * ih[p]), f);
                    }
                }
                if (a.Y.mode) f = fma((a.Y.p + (int64_t)a.Y.stride * e)[k], vol * (1.0 / NNODE), f);
            }
        }
        __builtin_amdgcn_sched_barrier(0);   // the next element's loads stay behind: half the registers
    }
    if (doS) asm_store<DIM, NB, SYM, TILE>(nd, acc, val, ld, zero);
    if (doF) rhs[nd.i * NB + k] += f;
}

// The Gauss sum of a group of coefficients: A alone (AGROUP), or B, C, D, X, Y
// (D alone: k_assemble_points).
// For each quadrature point the block stages its elements' points of the
// group in LDS (a thread per double, whole runs of a data point; zeros for
// elements outside the grid), and every node reads its 2^DIM elements from
// there (each double once per block and point instead of once per node
// through L1): B, C, D, X, Y of three equations on Brick 48x47x49 1.09 ->
// 1.00 ms, and with the next point fetched during the sums 0.77 ms (bytes
// alone 0.12 ms); C, D, Y of one on Brick 63x64x40 167 -> 94 us (bytes alone
// 13 us).  What is left is LDS reads and sums in turn with two barriers a point.
template <int DIM, int NB>
struct AsmBlock {
    static constexpr int ELEMENTS = asm_tile_elements(DIM, asm_nodes_per_wave<NB>());   // of the block, at most
    static constexpr int dpsA = NB * DIM * NB * DIM, dpsB = NB * DIM * NB, dpsD = NB * NB, dpsX = NB * DIM, dpsY = NB;
    // doubles per element of each group
    static constexpr int A_SIZE = dpsA, REST_SIZE = 2 * dpsB + dpsD + dpsX + dpsY;
};

// Grid index of each element of the block, -1 outside the grid.
template <int DIM, int NB, bool TILE>
__device__ __forceinline__ void asm_element_table(const AsmArgs& a, const AsmTile& tile, int64_t* index)
{
    const int wx = TILE ? tile.wx : asm_nodes_per_wave<NB>(), wy = TILE ? tile.wy : asm_wide_y(DIM),
              wz = TILE ? tile.wz : asm_wide_z(DIM);
    const int ex = wx + 1, ey = wy + 1,
              elements = TILE ? ex * ey * (DIM == 3 ? wz + 1 : 1) : AsmBlock<DIM, NB>::ELEMENTS;
    const int64_t bx = blockIdx.x % tile.gx, by = (blockIdx.x / tile.gx) % tile.gy,
                  bz = blockIdx.x / (tile.gx * tile.gy);
    for (int el = threadIdx.x; el < elements; el += kBlock) {
        const int64_t k0 = bx * wx - 1 + el % ex, k1 = by * wy - 1 + (el / ex) % ey,
                      k2 = DIM == 3 ? bz * wz - 1 + el / (ex * ey) : 0;
        const bool in = k0 >= 0 && k0 < a.ne0 && k1 >= 0 && k1 < a.ne1 && (DIM == 2 || (k2 >= 0 && k2 < a.ne2));
        index[el] = in ? k0 + (int64_t)a.ne0 * (k1 + (int64_t)a.ne1 * k2) : -1;
    }
}

template <int DIM, int NB, bool SYM, bool AGROUP, bool TILE>
__global__ __launch_bounds__(kBlock) void k_assemble_gauss(AsmArgs a, AsmTile tile, double* __restrict__ val,
                                                           int64_t ld, bool zero, double* __restrict__ rhs)
{
    using Blk = AsmBlock<DIM, NB>;
    constexpr int NS = StencilShape<DIM>::NS;
    constexpr int NNODE = 1 << DIM;
    constexpr int PER = AGROUP ? Blk::A_SIZE : Blk::REST_SIZE;
    constexpr int oB = 0, oC = Blk::dpsB, oD = 2 * Blk::dpsB, oX = oD + Blk::dpsD, oY = oX + Blk::dpsX;
    __shared__ double lds[Blk::ELEMENTS * PER];
    const AsmNode<DIM, NB, TILE> nd(a, tile);
    const int k = nd.k, m = nd.m;
    const int wx = TILE ? tile.wx : asm_nodes_per_wave<NB>(), wy = TILE ? tile.wy : asm_wide_y(DIM),
              wz = TILE ? tile.wz : asm_wide_z(DIM);
    const int ex = wx + 1, ey = wy + 1, elements = TILE ? ex * ey * (DIM == 3 ? wz + 1 : 1) : Blk::ELEMENTS;
    const double ih[3] = {1.0 / a.h0, 1.0 / a.h1, 1.0 / a.h2};
    double vol = a.h0 * a.h1;
    if (DIM == 3) vol *= a.h2;
    const bool doS = AGROUP || (a.B.mode | a.C.mode | a.D.mode) != 0;
    const bool doF = !AGROUP && rhs != nullptr && m == 0 && (a.X.mode | a.Y.mode) != 0;
    __shared__ int64_t index[Blk::ELEMENTS];
    asm_element_table<DIM, NB, TILE>(a, tile, index);
    __syncthreads();
    // the points of quadrature point q of one coefficient, DPS doubles each:
    // loaded into registers (ahead, see AHEAD), then stored
    auto fetch = [&](const CoefDev& c, auto& v, auto dps, int q) {
        constexpr int DPS = decltype(dps)::value;
        if (!c.mode) return;
        const int point = (AGROUP && c.iso) ? 1 : DPS;   // an isotropic A stages its scalar only
        const double* p = c.p + (c.mode == RG_COEF_EXPANDED ? q * point : 0);
        int tid = threadIdx.x;
        if (AGROUP || NB == 1) asm volatile("" : "+v"(tid));   // addresses formed anew for each point: registers
#pragma unroll
        for (int u = 0; u < (Blk::ELEMENTS * DPS + kBlock - 1) / kBlock; ++u) {
            const int idx = tid + u * kBlock, el = idx / DPS, o = idx % DPS;
            v[u] = 0.0;
            if (idx < elements * DPS && o < point) {
                const int64_t e = index[el];
                if (e >= 0) v[u] = p[e * c.stride + o];
            }
        }
    };
    auto store = [&](const CoefDev& c, const auto& v, auto dps, int offset) {
        constexpr int DPS = decltype(dps)::value;
        if (!c.mode) return;
#pragma unroll
        for (int u = 0; u < (Blk::ELEMENTS * DPS + kBlock - 1) / kBlock; ++u) {
            const int idx = threadIdx.x + u * kBlock;
            if (idx < elements * DPS) lds[idx / DPS * PER + offset + idx % DPS] = v[u];
        }
    };
    constexpr auto trips = [](int dps) { return (Blk::ELEMENTS * dps + kBlock - 1) / kBlock; };
    double fA[AGROUP ? trips(Blk::dpsA) : 1], fB[AGROUP ? 1 : trips(Blk::dpsB)], fC[AGROUP ? 1 : trips(Blk::dpsB)],
        fD[AGROUP ? 1 : trips(Blk::dpsD)], fX[AGROUP ? 1 : trips(Blk::dpsX)], fY[AGROUP ? 1 : trips(Blk::dpsY)];
    auto fetch_point = [&](int q) {
        if constexpr (AGROUP) {
            fetch(a.A, fA, IC<Blk::dpsA>{}, q);
        } else {
            fetch(a.B, fB, IC<Blk::dpsB>{}, q);
            fetch(a.C, fC, IC<Blk::dpsB>{}, q);
            fetch(a.D, fD, IC<Blk::dpsD>{}, q);
            fetch(a.X, fX, IC<Blk::dpsX>{}, q);
            fetch(a.Y, fY, IC<Blk::dpsY>{}, q);
        }
    };
    double acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s] = 0.0;
    double f = 0.0;
    const double w = vol / NNODE;
    const double g0 = 0.5 - 0.5 / 1.73205080756887719318, g1 = 0.5 + 0.5 / 1.73205080756887719318;
    const int e0 = nd.corner * PER;   // the node's first element in LDS
    // the next point's loads during the sums of this one: for systems other
    // than A (A's points beside its sums took more than 256 registers; a
    // single PDE's few doubles gain nothing: 94 -> 104 us)
    constexpr bool AHEAD = !AGROUP && NB > 1;
    if (AHEAD) fetch_point(0);
#pragma unroll 1
    for (int q = 0; q < NNODE; ++q) {
        __syncthreads();
        if (!AHEAD) fetch_point(q);
        if constexpr (AGROUP) {
            store(a.A, fA, IC<Blk::dpsA>{}, 0);
        } else {
            store(a.B, fB, IC<Blk::dpsB>{}, oB);
            store(a.C, fC, IC<Blk::dpsB>{}, oC);
            store(a.D, fD, IC<Blk::dpsD>{}, oD);
            store(a.X, fX, IC<Blk::dpsX>{}, oX);
            store(a.Y, fY, IC<Blk::dpsY>{}, oY);
        }
        __syncthreads();
        if (AHEAD && q + 1 < NNODE) fetch_point(q + 1);
        double phi[DIM][2];   // 1-D shape functions at the point
#pragma unroll
        for (int p = 0; p < DIM; ++p) {
            phi[p][1] = ((q >> p) & 1) ? g1 : g0;
            phi[p][0] = 1.0 - phi[p][1];
        }
        // N[b], and |dN_b/dx_p| by the bits of b along the other axes (its
        // sign is a compile-time one at each use)
        double N[NNODE], M[DIM][NNODE / 2];
#pragma unroll
        for (int b = 0; b < NNODE; ++b) {
            N[b] = 1.0;
#pragma unroll
            for (int p = 0; p < DIM; ++p) N[b] *= phi[p][(b >> p) & 1];
        }
#pragma unroll
        for (int p = 0; p < DIM; ++p)
#pragma unroll
            for (int r = 0; r < NNODE / 2; ++r) {
                const int o1 = p == 0 ? 1 : 0, o2 = p == 2 ? 1 : 2;
                M[p][r] = ih[p] * phi[o1][r & 1];
                if (DIM == 3) M[p][r] *= phi[DIM == 3 ? o2 : 0][r >> 1];
            }
        auto G = [&](int b, int p) {
            const int b1 = (b >> (p == 0 ? 1 : 0)) & 1, b2 = DIM == 3 ? (b >> (p == 2 ? 1 : 2)) & 1 : 0;
            const double g = M[p][b1 + 2 * b2];
            return ((b >> p) & 1) ? g : -g;
        };
#pragma unroll
        for (int t = 0; t < NNODE; ++t) {
            const double* P = lds + e0 + ((t & 1) + ex * (((t >> 1) & 1) + ey * (t >> 2))) * PER;
            const int la = (NNODE - 1) - t;   // the node's local index in element t
            double u[DIM], c0 = 0.0;
#pragma unroll
            for (int j = 0; j < DIM; ++j) u[j] = 0.0;
            if constexpr (AGROUP) {
                if (a.A.iso) {
#pragma unroll
                    for (int j = 0; j < DIM; ++j) u[j] = P[0] * G(la, j);
                } else {
#pragma unroll
                    for (int j = 0; j < DIM; ++j)
#pragma unroll
                        for (int p = 0; p < DIM; ++p)
                            u[j] = fma(P[k + NB * (p + DIM * (m + NB * j))], G(la, p), u[j]);
                }
            } else {
                if (a.C.mode) {
#pragma unroll
                    for (int j = 0; j < DIM; ++j) u[j] = P[oC + k + NB * (m + NB * j)] * N[la];
                }
                if (a.B.mode) {
#pragma unroll
                    for (int p = 0; p < DIM; ++p) c0 = fma(P[oB + k + NB * (p + DIM * m)], G(la, p), c0);
                }
                if (a.D.mode) c0 = fma(P[oD + k + NB * m], N[la], c0);
            }
            if (doS) {
#pragma unroll
                for (int b = 0; b < NNODE; ++b) {
                    const int s = asm_slot<DIM>(t, b);
                    if (SYM && s < StencilShape<DIM>::CENTER) continue;
                    double r = AGROUP ? acc[s] : fma(c0, N[b], acc[s]);
                    if (AGROUP || a.C.mode) {
#pragma unroll
                        for (int j = 0; j < DIM; ++j) r = fma(u[j], G(b, j), r);
                    }
                    acc[s] = r;
                }
            }
            if (doF) {
                if (a.X.mode) {
#pragma unroll
                    for (int p = 0; p < DIM; ++p) f = fma(P[oX + k + NB * p], G(la, p), f);
                }
                if (a.Y.mode) f = fma(P[oY + k], N[la], f);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (!nd.valid) return;
    if (doS) {
#pragma unroll
        for (int s = 0; s < NS; ++s) acc[s] *= w;
        asm_store<DIM, NB, SYM, TILE>(nd, acc, val, ld, zero);
    }
    if (doF) rhs[nd.i * NB + k] += w * f;
}

// The Gauss sum of D alone on quadrature points.  Its points of all the
// block's elements fit in the LDS at once, so they are staged in one go (whole
// runs of memory) and summed with constant weights N_a N_b: one barrier instead
// of two per point, which k_assemble_gauss shares among its coefficients and D
// alone did not repay (one equation, us per call, gather kernel with a thread
// per node / staged by points / here: 64x64x40 elements 70 / 77 / 50, 80x80x40
// 101 / 114 / 47, 128x64x32 100 / 111 / 45; four equations 16x20x20 61 / 77 / 52).
template <int DIM, int NB, bool SYM, bool TILE>
__global__ __launch_bounds__(kBlock) void k_assemble_points(AsmArgs a, AsmTile tile, double* __restrict__ val, int64_t ld,
                                                            bool zero)
{
    using Blk = AsmBlock<DIM, NB>;
    constexpr int NS = StencilShape<DIM>::NS, NNODE = 1 << DIM;
    constexpr int DPE = NNODE * Blk::dpsD, PER = DPE + 1;   // doubles per element; odd: lanes read different banks
    __shared__ double lds[Blk::ELEMENTS * PER];
    __shared__ int64_t index[Blk::ELEMENTS];
    const AsmNode<DIM, NB, TILE> nd(a, tile);
    const int ex = (TILE ? tile.wx : asm_nodes_per_wave<NB>()) + 1, ey = (TILE ? tile.wy : asm_wide_y(DIM)) + 1,
              elements = TILE ? ex * ey * (DIM == 3 ? tile.wz + 1 : 1) : Blk::ELEMENTS;
    asm_element_table<DIM, NB, TILE>(a, tile, index);
    __syncthreads();
    constexpr int TRIPS = (Blk::ELEMENTS * DPE + kBlock - 1) / kBlock;
    double v[TRIPS];
#pragma unroll
    for (int u = 0; u < TRIPS; ++u) {
        const int idx = threadIdx.x + u * kBlock;
        v[u] = 0.0;
        if (idx < elements * DPE) {
            const int64_t e = index[idx / DPE];
            if (e >= 0) v[u] = a.D.p[e * a.D.stride + idx % DPE];
        }
    }
#pragma unroll
    for (int u = 0; u < TRIPS; ++u) {
        const int idx = threadIdx.x + u * kBlock;
        if (idx < elements * DPE) lds[idx / DPE * PER + idx % DPE] = v[u];
    }
    __syncthreads();
    if (!nd.valid) return;
    constexpr double near = 0.5 + 0.5 / 1.73205080756887719318, far = 0.5 - 0.5 / 1.73205080756887719318;
    // N_b at point q: a factor per axis, by whether node and point agree on it
    auto N = [&](int b, int q) {
        double n = 1.0;
#pragma unroll
        for (int p = 0; p < DIM; ++p) n *= ((b ^ q) >> p) & 1 ? far : near;
        return n;
    };
    double acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s] = 0.0;
#pragma unroll
    for (int t = 0; t < NNODE; ++t) {
        const double* P = lds + (nd.corner + (t & 1) + ex * (((t >> 1) & 1) + ey * (t >> 2))) * PER + nd.k + NB * nd.m;
#pragma unroll
        for (int q = 0; q < NNODE; ++q) {
            const double c = P[q * Blk::dpsD] * N((NNODE - 1) - t, q);
#pragma unroll
            for (int b = 0; b < NNODE; ++b) {
                const int s = asm_slot<DIM>(t, b);
                if (SYM && s < StencilShape<DIM>::CENTER) continue;
                acc[s] = fma(c, N(b, q), acc[s]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    double w = a.h0 * a.h1 / NNODE;
    if (DIM == 3) w *= a.h2;
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s] *= w;
    asm_store<DIM, NB, SYM, TILE>(nd, acc, val, ld, zero);
}

// Element-constant isotropic A = kappa_e I (single PDE, full quadrature),
// optionally with element-constant Y and no other coefficient: the
// reference's constant-coefficient branch (DefaultAssembler3D.cpp:906-993,
// load :2205-2214; DefaultAssembler2D.cpp:301-326, :578-583).  The element
// matrix is then kappa_e K with K(a, b) = sum_d s_d(a, b) / h_d
// prod_{o != d} h_o m_o(a, b), s = +1 / -1 and m = 1/3 / 1/6 for equal /
// different local coordinates along an axis (the 2-point Gauss rule
// integrates these products exactly), so K depends only on which axes a and
// b agree in: kt[bit d set = agree along d] (2^DIM values, from the host).
// One thread per node gathers the 2^DIM elements around it; each value slot
// is written once (plainly when the matrix is known to hold zeros, ZERO),
// and Y contributes Y_e vol / 2^DIM to the node's rhs.
struct IsoArgs {
    const double* kappa;
    int64_t kstride;       // doubles between elements' kappa (0: one value for all)
    const double* Y;
    int64_t ystride;
    int64_t n0, n1, n2;
    int ne0, ne1, ne2;
    double kt[8];
    double fy;             // vol / 2^DIM
};

template <int DIM, bool SYM, bool ZERO>
__global__ __launch_bounds__(kBlock) void k_assemble_iso(IsoArgs a, double* __restrict__ val, int64_t ld, int64_t N,
                                                         double* __restrict__ rhs)
{
    constexpr int NS = StencilShape<DIM>::NS;
    constexpr int CEN = StencilShape<DIM>::CENTER;
    constexpr int NST = stored_slots<DIM, SYM>();
    constexpr int FIRST = SYM ? CEN : 0;
    constexpr int NNODE = 1 << DIM;
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= N) return;
    const int64_t x = i % a.n0, y = (i / a.n0) % a.n1, z = (DIM == 3) ? i / (a.n0 * a.n1) : 0;
    double kap[NNODE];
#pragma unroll
    for (int e = 0; e < NNODE; ++e) {
        const int ex = e & 1, ey = (e >> 1) & 1, ez = (e >> 2) & 1;
        const int64_t k0 = x - 1 + ex, k1 = y - 1 + ey, k2 = (DIM == 3) ? z - 1 + ez : 0;
        const bool in = k0 >= 0 && k0 < a.ne0 && k1 >= 0 && k1 < a.ne1 && (DIM == 2 || (k2 >= 0 && k2 < a.ne2));
        const int64_t el = in ? k0 + (int64_t)a.ne0 * (k1 + (int64_t)a.ne1 * k2) : 0;
        kap[e] = in ? a.kappa[a.kstride * el] : 0.0;
    }
    double acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s] = 0.0;
    // element e = (ex, ey, ez) holds node i at local bits (1-ex, 1-ey, 1-ez);
    // local node b of e is the neighbour at offset (ex+b0-1, ey+b1-1, ez+b2-1)
#pragma unroll
    for (int e = 0; e < NNODE; ++e) {
#pragma unroll
        for (int b = 0; b < NNODE; ++b) {
            const int agree = ((b & 1) == 1 - (e & 1) ? 1 : 0) | (((b >> 1) & 1) == 1 - ((e >> 1) & 1) ? 2 : 0) |
                              (DIM == 3 && ((b >> 2) & 1) == 1 - ((e >> 2) & 1) ? 4 : 0);
            const int s = ((e & 1) + (b & 1)) + 3 * (((e >> 1) & 1) + ((b >> 1) & 1)) +
                          (DIM == 3 ? 9 * (((e >> 2) & 1) + ((b >> 2) & 1)) : 0);
            acc[s] = fma(kap[e], a.kt[agree], acc[s]);
        }
    }
#pragma unroll
    for (int t = 0; t < NST; ++t) {
        double* p = &val[(int64_t)t * ld + i];
        *p = ZERO ? acc[FIRST + t] : *p + acc[FIRST + t];
    }
    if (rhs && a.Y) {
        double f = 0.0;
#pragma unroll
        for (int e = 0; e < NNODE; ++e) {
            const int ex = e & 1, ey = (e >> 1) & 1, ez = (e >> 2) & 1;
            const int64_t k0 = x - 1 + ex, k1 = y - 1 + ey, k2 = (DIM == 3) ? z - 1 + ez : 0;
            const bool in = k0 >= 0 && k0 < a.ne0 && k1 >= 0 && k1 < a.ne1 && (DIM == 2 || (k2 >= 0 && k2 < a.ne2));
            const int64_t el = in ? k0 + (int64_t)a.ne0 * (k1 + (int64_t)a.ne1 * k2) : 0;
            f += in ? a.Y[a.ystride * el] * a.fy : 0.0;
        }
        rhs[i] += f;
    }
}

// Boundary terms, colour free: one thread per (node i, equation k,
// component m) visits the face elements around node i on every face of the
// domain the node lies on and adds row a (node i's local face index) of
//   EM_S[k,m,a,b] = sum_q w d[k + n m] N_a N_b,   EM_F[k,a] = sum_q w y[k] N_a
// -- the face integrals of DefaultAssembler2D/3D::assemblePDEBoundarySingle/
// System (2-point Gauss rule along each tangential axis, weight face measure
// / points; DefaultAssembler2D.cpp:601-840, DefaultAssembler3D.cpp:2233-2890)
// or, reduced, the one-point rule at the face centre (:1014-1200,
// :3274-3630).  Face elements are indexed as the reference's
// FunctionOnBoundary samples: faces x0=0, x0=L, x1=0, x1=L[, x2=0, x2=L],
// within a face the lower tangential element index fastest (m_faceOffset).
struct BndArgs {
    CoefDev d, y;
    int64_t n[3];        // nodes per axis
    int ne[3];           // elements per axis
    double h[3];
    int64_t face_off[6];
    int reduced;
};

template <int DIM, int NB, bool SYM>
__global__ __launch_bounds__(kBlock) void k_assemble_boundary(BndArgs a, double* __restrict__ val, int64_t ld,
                                                              int64_t N, double* __restrict__ rhs)
{
    constexpr int NS = StencilShape<DIM>::NS;
    constexpr int CEN = StencilShape<DIM>::CENTER;
    constexpr int NST = stored_slots<DIM, SYM>();
    constexpr int FIRST = SYM ? CEN : 0;
    constexpr int NFN = 1 << (DIM - 1);                // nodes per face element
    const int km = blockIdx.y;
    const int k = km % NB, m = km / NB;
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= N) return;
    const int64_t c[3] = {i % a.n[0], (i / a.n[0]) % a.n[1], DIM == 3 ? i / (a.n[0] * a.n[1]) : 0};
    const bool doS = a.d.mode != 0;
    const bool doF = rhs != nullptr && m == 0 && a.y.mode != 0;
    const int nq = a.reduced ? 1 : NFN;
    const double g0 = 0.5 - 0.5 / 1.73205080756887719318, g1 = 0.5 + 0.5 / 1.73205080756887719318;
    double acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s] = 0.0;
    double f = 0.0;
    bool any = false;
#pragma unroll
    for (int face = 0; face < 2 * DIM; ++face) {
        const int ax = face / 2, side = face % 2;
        if (c[ax] != (side ? a.n[ax] - 1 : 0)) continue;
        any = true;
        const int t0 = (ax == 0) ? 1 : 0;
        const int t1 = (DIM == 3) ? ((ax == 2) ? 1 : 2) : -1;
        const double meas = a.h[t0] * (DIM == 3 ? a.h[t1] : 1.0);
        const double w = meas / nq;
#pragma unroll
        for (int e1 = 0; e1 < (DIM == 3 ? 2 : 1); ++e1)
#pragma unroll
            for (int e0 = 0; e0 < 2; ++e0) {
                const int64_t j0 = c[t0] - 1 + e0;
                const int64_t j1 = (DIM == 3) ? c[t1] - 1 + e1 : 0;
                if (j0 < 0 || j0 >= a.ne[t0]) continue;
                if (DIM == 3 && (j1 < 0 || j1 >= a.ne[t1])) continue;
                const int64_t fe = a.face_off[face] + j0 + (int64_t)a.ne[t0] * j1;
                const int ab0 = 1 - e0, ab1 = 1 - e1;      // node i's local face bits
                for (int q = 0; q < nq; ++q) {
                    const double xi0 = a.reduced ? 0.5 : ((q & 1) ? g1 : g0);
                    const double xi1 = a.reduced ? 0.5 : (((q >> 1) & 1) ? g1 : g0);
                    const double Na = (ab0 ? xi0 : 1.0 - xi0) * (DIM == 3 ? (ab1 ? xi1 : 1.0 - xi1) : 1.0);
                    if (doS) {
                        const double dv = coef_pt(a.d, fe, q, NB * NB)[k + NB * m];
#pragma unroll
                        for (int b = 0; b < NFN; ++b) {
                            const int bb0 = b & 1, bb1 = (b >> 1) & 1;
                            const double Nb = (bb0 ? xi0 : 1.0 - xi0) * (DIM == 3 ? (bb1 ? xi1 : 1.0 - xi1) : 1.0);
                            int off[3] = {1, 1, 1};
                            off[t0] = e0 + bb0;
                            if (DIM == 3) off[t1] = e1 + bb1;
                            const int s = off[0] + 3 * off[1] + (DIM == 3 ? 9 * off[2] : 0);
                            acc[s] += w * dv * Na * Nb;
                        }
                    }
                    if (doF) f += w * coef_pt(a.y, fe, q, NB)[k] * Na;
                }
            }
    }
    if (!any) return;
    if (doS) {
#pragma unroll
        for (int t = 0; t < NST; ++t)
            val[(int64_t)(t * NB * NB + k + NB * m) * ld + i] += acc[FIRST + t];
    }
    if (doF) rhs[i * NB + k] += f;
}

// Dirac points in order (RipleyDomain::assemblePDEDirac, RipleyDomain.cpp:
// 1756-1800): rhs[k + n*node] += y[p][k]; diagonal block += d[p] (k + n*m).
template <int NB>
__global__ void k_add_dirac(int64_t count, const int64_t* __restrict__ nodes, const double* __restrict__ d,
                            const double* __restrict__ y, double* __restrict__ val, int64_t ld, int diag_slot,
                            double* __restrict__ rhs)
{
    if (threadIdx.x >= NB * NB) return;
    const int k = threadIdx.x % NB, m = threadIdx.x / NB;
    for (int64_t p = 0; p < count; ++p) {
        const int64_t i = nodes[p];
        if (d) val[(int64_t)(diag_slot * NB * NB + k + NB * m) * ld + i] += d[p * NB * NB + k + NB * m];
        if (y && rhs && m == 0) rhs[i * NB + k] += y[p * NB + k];
    }
}

void launch_assemble_boundary(rg_matrix* m, const rg_coef* d, const rg_coef* y, int reduced, double* rhs)
{
    const Geom& g = m->g;
    auto cv = [](const rg_coef* x) {
        return x ? CoefDev{x->data, x->data ? x->mode : 0, x->elem_stride, 0} : CoefDev{nullptr, 0, 0, 0};
    };
    BndArgs a;
    a.d = cv(d);
    a.y = cv(y);
    for (const rg_coef* x : {d, y}) {
        if (!x) continue;
        RG_CHECK(x->mode >= RG_COEF_EMPTY && x->mode <= RG_COEF_EXPANDED, RG_VALUE_ERROR,
                 "assemble_boundary: unknown coefficient mode");
        RG_CHECK(x->mode == RG_COEF_EMPTY || x->data != nullptr, RG_VALUE_ERROR,
                 "assemble_boundary: coefficient data is NULL");
        RG_CHECK(!(reduced && x->mode == RG_COEF_EXPANDED), RG_VALUE_ERROR,
                 "assemble_boundary: reduced-order coefficients cannot be expanded");
        RG_CHECK(!x->isotropic, RG_VALUE_ERROR, "assemble_boundary: isotropic is defined for A only");
    }
    for (int t = 0; t < 3; ++t) {
        a.n[t] = g.nn[t];
        a.ne[t] = g.ne[t];
        a.h[t] = g.h[t];
    }
    int64_t off = 0;
    for (int f = 0; f < 6; ++f) {
        a.face_off[f] = off;
        if (f >= 2 * g.dim) continue;
        const int ax = f / 2;
        int64_t cnt = 1;
        for (int t = 0; t < g.dim; ++t)
            if (t != ax) cnt *= g.ne[t];
        off += cnt;
    }
    a.reduced = reduced;
    if (!a.d.mode && !(a.y.mode && rhs)) return;
    const dim3 grid((unsigned)((g.N + kBlock - 1) / kBlock), (unsigned)(g.bs * g.bs));
    dispatch(g, m->symmetric, [&](auto D, auto B, auto S) {
        hipLaunchKernelGGL((k_assemble_boundary<D.value, B.value, S.value>), grid, dim3(kBlock), 0, m->ctx->stream, a,
                           m->val, g.ld, g.N, rhs);
    });
    RG_HIP(hipGetLastError());
    m->val32_valid = false;
    if (a.d.mode) m->val_zero = false;
}

void launch_add_dirac(rg_matrix* m, int64_t count, const int64_t* d_nodes, const double* d_d, const double* d_y,
                      double* rhs)
{
    const Geom& g = m->g;
    const int diag_slot = m->symmetric ? 0 : (g.dim == 3 ? 13 : 4);
    dispatch_bs(g.bs, [&](auto B) {
        hipLaunchKernelGGL((k_add_dirac<B.value>), dim3(1), dim3(64), 0, m->ctx->stream, count, d_nodes, d_d, d_y,
                           m->val, g.ld, diag_slot, rhs);
    });
    RG_HIP(hipGetLastError());
    m->val32_valid = false;
    if (d_d) m->val_zero = false;
}

void launch_assemble(rg_matrix* m, const rg_pde_coefs& c, int reduced, double* rhs)
{
    const Geom& g = m->g;
    AsmArgs a;
    auto cv = [](const rg_coef& x) { return CoefDev{x.data, x.data ? x.mode : 0, x.elem_stride, x.isotropic}; };
    a.A = cv(c.A); a.B = cv(c.B); a.C = cv(c.C); a.D = cv(c.D); a.X = cv(c.X); a.Y = cv(c.Y);
    const rg_coef* all[6] = {&c.A, &c.B, &c.C, &c.D, &c.X, &c.Y};
    for (int t = 0; t < 6; ++t) {
        const rg_coef& x = *all[t];
        RG_CHECK(x.mode >= RG_COEF_EMPTY && x.mode <= RG_COEF_EXPANDED, RG_VALUE_ERROR,
                 "assemble: unknown coefficient mode");
        RG_CHECK(x.mode == RG_COEF_EMPTY || x.data != nullptr, RG_VALUE_ERROR,
                 "assemble: coefficient data is NULL");
        RG_CHECK(!(reduced && x.mode == RG_COEF_EXPANDED), RG_VALUE_ERROR,
                 "assemble: reduced-order coefficients cannot be expanded");
    }
    RG_CHECK(!c.A.isotropic || g.bs == 1, RG_VALUE_ERROR,
             "assemble: isotropic A is defined for a single PDE only");
    a.n0 = g.nn[0]; a.n1 = g.nn[1]; a.n2 = g.nn[2];
    a.ne0 = g.ne[0]; a.ne1 = g.ne[1]; a.ne2 = g.ne[2];
    a.h0 = g.h[0]; a.h1 = g.h[1]; a.h2 = g.h[2];
    const bool iso_const = g.bs == 1 && !reduced && c.A.mode == RG_COEF_ELEMENT && c.A.isotropic && c.A.data &&
                           !c.B.mode && !c.C.mode && !c.D.mode && !c.X.mode &&
                           (c.Y.mode == RG_COEF_EMPTY || c.Y.mode == RG_COEF_ELEMENT);
    if (iso_const) {
        IsoArgs ia;
        ia.kappa = c.A.data;
        ia.kstride = c.A.elem_stride;
        ia.Y = (c.Y.mode == RG_COEF_ELEMENT) ? c.Y.data : nullptr;
        ia.ystride = c.Y.elem_stride;
        ia.n0 = g.nn[0]; ia.n1 = g.nn[1]; ia.n2 = g.nn[2];
        ia.ne0 = g.ne[0]; ia.ne1 = g.ne[1]; ia.ne2 = g.ne[2];
        double vol = 1.0;
        for (int d = 0; d < g.dim; ++d) vol *= g.h[d];
        ia.fy = vol / (1 << g.dim);
        // K(agree) = sum_d s_d / h_d prod_{o != d} h_o m_o
        for (int ag = 0; ag < (1 << g.dim); ++ag) {
            double kt = 0.0;
            for (int d = 0; d < g.dim; ++d) {
                double t = (((ag >> d) & 1) ? 1.0 : -1.0) / g.h[d];
                for (int o = 0; o < g.dim; ++o)
                    if (o != d) t *= g.h[o] * (((ag >> o) & 1) ? 1.0 / 3.0 : 1.0 / 6.0);
                kt += t;
            }
            ia.kt[ag] = kt;
        }
        for (int ag = 1 << g.dim; ag < 8; ++ag) ia.kt[ag] = 0.0;
        const dim3 grid((unsigned)((g.N + kBlock - 1) / kBlock));
        auto go = [&](auto D, auto S, auto Z) {
            hipLaunchKernelGGL((k_assemble_iso<D.value, S.value, Z.value>), grid, dim3(kBlock), 0, m->ctx->stream, ia,
                               m->val, g.ld, g.N, rhs);
        };
        auto byz = [&](auto D, auto S) {
            if (m->val_zero) go(D, S, BC<true>{});
            else go(D, S, BC<false>{});
        };
        if (g.dim == 3) {
            if (m->symmetric) byz(IC<3>{}, BC<true>{});
            else byz(IC<3>{}, BC<false>{});
        } else {
            if (m->symmetric) byz(IC<2>{}, BC<true>{});
            else byz(IC<2>{}, BC<false>{});
        }
    } else {
        // the coefficients of each kernel (k_assemble_const, k_assemble_gauss)
        AsmArgs ac = a, ag = a;
        CoefDev* const both[6][2] = {{&ac.A, &ag.A}, {&ac.B, &ag.B}, {&ac.C, &ag.C},
                                     {&ac.D, &ag.D}, {&ac.X, &ag.X}, {&ac.Y, &ag.Y}};
        bool is_const = false;
        for (auto& p : both) {
            const int mode = p[0]->mode;
            const bool cst = mode == RG_COEF_ELEMENT;
            is_const = is_const || cst;
            p[cst ? 1 : 0]->mode = RG_COEF_EMPTY;
        }
        dispatch(g, m->symmetric, [&](auto D, auto B, auto S) {
            constexpr int npw = asm_nodes_per_wave<B.value>();
            // f(TILE, tile, grid) with the tile of the closed form (0) or of the staged sums (1)
            auto with_tile = [&](int staged, auto&& f) {
                AsmTile& t = m->asm_tile[staged];
                if (!t.wx) t = asm_tile(D.value, g.nn, npw, staged);
                RG_CHECK(t.gx * t.gy * t.gz < ((int64_t)1 << 31), RG_VALUE_ERROR, "assemble: grid too large");
                const dim3 grid((unsigned)(t.gx * t.gy * t.gz));
                if (asm_is_wide(t, D.value, npw)) f(BC<false>{}, t, grid);
                else f(BC<true>{}, t, grid);
            };
            bool zero = m->val_zero;
            if (is_const) {
                with_tile(0, [&](auto T, const AsmTile& t, dim3 grid) {
                    auto go = [&](auto One) {
                        hipLaunchKernelGGL((k_assemble_const<D.value, B.value, S.value, One.value, T.value>), grid,
                                           dim3(kBlock), 0, m->ctx->stream, ac, t, m->val, g.ld, zero, rhs);
                    };
                    if (reduced) go(BC<true>{});
                    else go(BC<false>{});
                });
                if (ac.A.mode || ac.B.mode || ac.C.mode || ac.D.mode) zero = false;
            }
            auto gauss = [&](auto AGroup) {
                with_tile(1, [&](auto T, const AsmTile& t, dim3 grid) {
                    hipLaunchKernelGGL((k_assemble_gauss<D.value, B.value, S.value, AGroup.value, T.value>), grid,
                                       dim3(kBlock), 0, m->ctx->stream, ag, t, m->val, g.ld, zero, rhs);
                });
            };
            if (ag.A.mode) {
                gauss(BC<true>{});
                zero = false;
            }
            if (ag.D.mode && !(ag.B.mode || ag.C.mode || ag.X.mode || ag.Y.mode))
                with_tile(1, [&](auto T, const AsmTile& t, dim3 grid) {
                    hipLaunchKernelGGL((k_assemble_points<D.value, B.value, S.value, T.value>), grid, dim3(kBlock), 0,
                                       m->ctx->stream, ag, t, m->val, g.ld, zero);
                });
            else if (ag.B.mode || ag.C.mode || ag.D.mode || ag.X.mode || ag.Y.mode)
                gauss(BC<false>{});
        });
    }
    RG_HIP(hipGetLastError());
    m->val32_valid = false;
    if (c.A.mode || c.B.mode || c.C.mode || c.D.mode) m->val_zero = false;
}

// -------------------------------------------------------------------- SpMV
// paso SystemMatrix::MatrixVector -> SparseMatrix_MatrixVector_CSR_OFFSET0
// (paso/src/SparseMatrix_MatrixVector.cpp:191-336): out = alpha*A*in +
// beta*out, out first scaled by beta (zeroed for beta == 0).  BETA selects
// the epilogue at compile time (0: beta == 0, 1: beta == 1, 2: general): a
// run-time branch on beta inside the row loop cost 150 registers.
template <int DIM, int BS, bool SYM, typename VT, int BETA>
__global__ __launch_bounds__(kBlock) void k_spmv(const VT* __restrict__ val, int64_t ld, int64_t N,
                                                 int64_t s1, int64_t s2, int64_t chunk,
                                                 const double* __restrict__ x, double* __restrict__ y,
                                                 double alpha, double beta)
{
    const RowRange rr = block_rows(N, chunk);
    stencil_block<DIM, BS, SYM, VT>(val, ld, N, s1, s2, rr.r0, rr.r1, x, [&](int64_t i, const double (&acc)[BS]) {
#pragma unroll
        for (int r = 0; r < BS; ++r) {
            if (BETA == 0) y[i * BS + r] = alpha * acc[r];
            else if (BETA == 1) y[i * BS + r] = fma(alpha, acc[r], y[i * BS + r]);
            else y[i * BS + r] = fma(alpha, acc[r], beta * y[i * BS + r]);
        }
    });
}

void launch_spmv(rg_matrix* m, double alpha, const double* x, double beta, double* y)
{
    launch_spmv_on(m, alpha, x, beta, y, m->ctx->stream);
}

void launch_spmv_on(rg_matrix* m, double alpha, const double* x, double beta, double* y, hipStream_t st)
{
    const Geom& g = m->g;
    const Launch L = chunked_launch(g.N, spmv_rows_per_thread<double>());
    dispatch(g, m->symmetric, [&](auto D, auto B, auto S) {
        if (beta == 0.0)
            hipLaunchKernelGGL((k_spmv<D.value, B.value, S.value, double, 0>), dim3(L.grid), dim3(kBlock), 0,
                               st, m->val, g.ld, g.N, g.s1, g.s2, L.chunk, x, y, alpha, beta);
        else if (beta == 1.0)
            hipLaunchKernelGGL((k_spmv<D.value, B.value, S.value, double, 1>), dim3(L.grid), dim3(kBlock), 0,
                               st, m->val, g.ld, g.N, g.s1, g.s2, L.chunk, x, y, alpha, beta);
        else
            hipLaunchKernelGGL((k_spmv<D.value, B.value, S.value, double, 2>), dim3(L.grid), dim3(kBlock), 0,
                               st, m->val, g.ld, g.N, g.s1, g.s2, L.chunk, x, y, alpha, beta);
    });
    RG_HIP(hipGetLastError());
}

void launch_spmv32(rg_matrix* m, const double* x, double* y)
{
    const Geom& g = m->g;
    const Launch L = chunked_launch(g.N, spmv_rows_per_thread<float>());
    dispatch(g, m->symmetric, [&](auto D, auto B, auto S) {
        hipLaunchKernelGGL((k_spmv<D.value, B.value, S.value, float, 0>), dim3(L.grid), dim3(kBlock), 0,
                           m->ctx->stream, m->val32, g.ld, g.N, g.s1, g.s2, L.chunk, x, y, 1.0, 0.0);
    });
    RG_HIP(hipGetLastError());
}

// ---------------------------------------------------------------- nullify
// SparseMatrix::nullifyRowsAndCols_CSR(_BLK1) (paso/src/SparseMatrix.h:
// 494-535): a(i r, j c) := (i r == j c ? mdv : 0) where row_mask[i r] > 0 or
// col_mask[j c] > 0, over the PASO pattern.  With symmetric storage the two
// masks must be equal (checked by k_mask_differs).
template <int DIM, int BS, bool SYM>
__global__ __launch_bounds__(kBlock) void k_nullify(double* __restrict__ val, int64_t ld, int64_t N,
                                                    int64_t n0, int64_t n1, int64_t n2,
                                                    const double* __restrict__ mrow,
                                                    const double* __restrict__ mcol, double mdv)
{
    constexpr int NST = stored_slots<DIM, SYM>();
    constexpr int FIRST = SYM ? StencilShape<DIM>::CENTER : 0;
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= N) return;
    const int64_t x = i % n0, y = (i / n0) % n1, z = i / (n0 * n1);
    bool anyrow = false;
    double mr[BS];
#pragma unroll
    for (int r = 0; r < BS; ++r) {
        mr[r] = mrow[i * BS + r];
        anyrow |= mr[r] > 0.0;
    }
#pragma unroll
    for (int t = 0; t < NST; ++t) {
        const int s = FIRST + t;
        if (!slot_in_grid<DIM>(s, x, y, z, n0, n1, n2)) continue;
        int dx, dy, dz;
        slot_delta<DIM>(s, dx, dy, dz);
        const int64_t j = i + dx + dy * n0 + dz * n0 * n1;
        bool anycol = false;
        double mc[BS];
#pragma unroll
        for (int c = 0; c < BS; ++c) {
            mc[c] = mcol[j * BS + c];
            anycol |= mc[c] > 0.0;
        }
        if (!anyrow && !anycol) continue;
#pragma unroll
        for (int c = 0; c < BS; ++c)
#pragma unroll
            for (int r = 0; r < BS; ++r)
                if (mr[r] > 0.0 || mc[c] > 0.0)
                    val[(int64_t)(t * BS * BS + r + BS * c) * ld + i] = (j == i && r == c) ? mdv : 0.0;
    }
}

__global__ void k_mask_differs(const double* a, const double* b, int64_t n, int* flag)
{
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        if ((a[i] > 0.0) != (b[i] > 0.0)) *flag = 1;
}

void launch_nullify(rg_matrix* m, const double* row_mask, const double* col_mask, double mdv, int* d_flag)
{
    const Geom& g = m->g;
    const int grid = (int)((g.N + kBlock - 1) / kBlock);
    if (m->symmetric && row_mask != col_mask) {
        hipLaunchKernelGGL(k_mask_differs, dim3(std::min(grid, 1024)), dim3(kBlock), 0, m->ctx->stream,
                           row_mask, col_mask, g.N * g.bs, d_flag);
        RG_HIP(hipGetLastError());
        int h = 0;
        RG_HIP(hipMemcpyAsync(&h, d_flag, sizeof(int), hipMemcpyDeviceToHost, m->ctx->stream));
        RG_HIP(hipStreamSynchronize(m->ctx->stream));
        RG_CHECK(h == 0, RG_VALUE_ERROR,
                 "nullifyRowsAndCols: a matrix with symmetric storage needs equal row and column masks");
    }
    dispatch(g, m->symmetric, [&](auto D, auto B, auto S) {
        hipLaunchKernelGGL((k_nullify<D.value, B.value, S.value>), dim3(grid), dim3(kBlock), 0,
                           m->ctx->stream, m->val, g.ld, g.N, g.nn[0], g.nn[1], g.nn[2], row_mask,
                           col_mask, mdv);
    });
    RG_HIP(hipGetLastError());
    m->val32_valid = false;
    m->val_zero = false;
}

// ------------------------------------------------------------- CSR export
// The PASO main block in CSR form: row i lists its in-grid neighbours in
// ascending order (ripley/src/Brick.cpp:3000-3061) with the block values
// val[k*bs*bs + ir + bs*ic] (paso/src/SystemMatrix.h:404-492).
template <int DIM, int BS, bool SYM>
__global__ __launch_bounds__(kBlock) void k_export_csr(const double* __restrict__ val, int64_t ld,
                                                       int64_t N, int64_t n0, int64_t n1, int64_t n2,
                                                       const int32_t* __restrict__ ptr,
                                                       int32_t* __restrict__ index,
                                                       double* __restrict__ out)
{
    constexpr int NS = StencilShape<DIM>::NS;
    constexpr int C = StencilShape<DIM>::CENTER;
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= N) return;
    const int64_t x = i % n0, y = (i / n0) % n1, z = i / (n0 * n1);
    int64_t k = ptr[i];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if (!slot_in_grid<DIM>(s, x, y, z, n0, n1, n2)) continue;
        int dx, dy, dz;
        slot_delta<DIM>(s, dx, dy, dz);
        const int64_t j = i + dx + dy * n0 + dz * n0 * n1;
        if (index) index[k] = (int32_t)j;
        if (out) {
#pragma unroll
            for (int c = 0; c < BS; ++c)
#pragma unroll
                for (int r = 0; r < BS; ++r) {
                    double v;
                    if (!SYM || s >= C)
                        v = val[(int64_t)((SYM ? s - C : s) * BS * BS + r + BS * c) * ld + i];
                    else
                        v = val[(int64_t)((C - s) * BS * BS + c + BS * r) * ld + j];
                    out[k * BS * BS + r + BS * c] = v;
                }
        }
        ++k;
    }
}

void launch_export_csr_values(rg_matrix* m, const int32_t* d_ptr, int32_t* d_index, double* d_val)
{
    const Geom& g = m->g;
    const int grid = (int)((g.N + kBlock - 1) / kBlock);
    dispatch(g, m->symmetric, [&](auto D, auto B, auto S) {
        hipLaunchKernelGGL((k_export_csr<D.value, B.value, S.value>), dim3(grid), dim3(kBlock), 0,
                           m->ctx->stream, m->val, g.ld, g.N, g.nn[0], g.nn[1], g.nn[2], d_ptr,
                           d_index, d_val);
    });
    RG_HIP(hipGetLastError());
}

// ---------------------------------------------------------- FP32 values
__global__ void k_to_fp32(const double* __restrict__ a, float* __restrict__ b, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        b[i] = (float)a[i];
}

void launch_to_fp32(rg_matrix* m)
{
    const Geom& g = m->g;
    const int64_t n = (int64_t)g.nstore * g.bs * g.bs * g.ld;
    hipLaunchKernelGGL(k_to_fp32, dim3(4096), dim3(kBlock), 0, m->ctx->stream, m->val, m->val32, n);
    RG_HIP(hipGetLastError());
}

// ----------------------------------------------------------- host pattern
void csr_row_ptr(const Geom& g, int32_t* ptr)
{
    const int64_t n0 = g.nn[0], n1 = g.nn[1], n2 = g.nn[2];
    ptr[0] = 0;
    int64_t acc = 0;
    for (int64_t i = 0; i < g.N; ++i) {
        const int64_t x = i % n0, y = (i / n0) % n1, z = i / (n0 * n1);
        const int cx = 1 + (x > 0) + (x < n0 - 1);
        const int cy = 1 + (y > 0) + (y < n1 - 1);
        const int cz = (g.dim == 3) ? 1 + (z > 0) + (z < n2 - 1) : 1;
        acc += cx * cy * cz;
        ptr[i + 1] = (int32_t)acc;
    }
}

int64_t csr_nnz(const Geom& g)
{
    int64_t n = 1;
    for (int d = 0; d < g.dim; ++d) n *= 3 * g.nn[d] - 2;
    return n;
}

}  // namespace rg
