// Immersed-boundary coupling on gfx950.
//
// Per coupled step (the IBM functional of the reference,
// src/fsi/DataProcessors.hh:94-108, preceded by the progs' computeVelocity
// and force reset):
//   bin      every vertex's delta-kernel stencil into the lists of the 4x4x4
//            lattice tiles it touches, in one pass (a workgroup counts its
//            pairs per tile in LDS and reserves a run in each list), and a
//            copy of its position;
//   forces   per element (triangle / link / pair) contributions, then a
//            per-vertex gather over the CSR incidence lists (K5, no atomics);
//   stage    u = j/rho + F/2 on the cells of the touched tiles (from the
//            post-stream populations and the force of the last collision);
//   spread   a wave per touched tile, a workgroup for a long list: the list
//            put in vertex order, the tile's g + sum_k phi F_k a product of
//            matrix instructions over it (K6, deterministic, no float
//            atomics);
//   interp   U_k = sum phi phi phi u, sixteen lanes per vertex (four for the
//            top hat), each along x, and a butterfly (K4), fused with the
//            advection x += U;
//   move     per-particle area / volume / COM in FP64 with a
//            fixed reduction order, COM mapped onto the periodic grid (K7);
//   voxelize z-ray hits toggle a bit per column and node, parity fill of
//            the phase (K8), only when the inner and outer viscosities differ.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <initializer_list>
#include <string>
#include <type_traits>
#include <vector>

#include "ibm.hpp"
#include "interactions.hpp"
#include "lattice_dev.hpp"
#include "walls.hpp"

namespace bl {

namespace {

constexpr int kGeomSums = 5;       // a particle's geometry: area, volume, centroid
constexpr int kTileCap = 512;      // list entries per 4x4x4 tile (stencils touching it)
constexpr int kSmallTile = 128;    // the most entries of a tile that one wave spreads (kSparseTile below)
constexpr int kSparseTile = 64;    // the same where few tiles are touched: the others' waves are idle
constexpr int kMaxList = kTileCap; // entries the spreading kernel sorts in LDS
static_assert(kMaxList >= 4 * kSmallTile, "four waves of small tiles order their keys there");

// ------------------------------------------------------------- helpers
// Vertex data (positions, velocities, forces, element forces, stencil
// weights, spreading sums) is held and computed in the real type R: double
// with FP64 populations, float with FP32 and FP16-shifted ones.  Rest
// geometry, per-particle area / volume / centroid reductions and the
// conservation sums stay FP64 in both.

// Delta kernels (src/fsi/Dirac.h:23-66,74-101), 1-D factor; the branch is
// taken on the square root's argument, so that a lane forms one root.
template <class R>
__device__ __forceinline__ R dirac(int kernel, R x)
{
    const R dx = fabs(x);
    if (kernel == BL_KERNEL_ROMA) {
        const bool far = dx > R(0.5);
        const R q = sqrt(far ? -R(3) * (R(1) - dx) * (R(1) - dx) + R(1) : R(1) - R(3) * dx * dx);
        return (R(1.0) / R(6.0)) * (far ? (R(5.0) - R(3) * dx - q) : R(2.0) * (R(1) + q));
    }
    if (kernel == BL_KERNEL_PESKIN) {
        const bool near = dx <= R(1);
        const R q = sqrt(near ? R(1) + R(4) * dx * (R(1) - dx) : -R(7) + R(4) * dx * (R(3) - dx));
        return R(0.125) * (near ? (R(3) - R(2) * dx + q) : (R(5) - R(2) * dx - q));
    }
    return R(1.) - fabs(x);
}

__device__ __forceinline__ int wrap_node(int i, int n, int per)
{
    if (per) {
        int r = i % n;
        return r < 0 ? r + n : r;
    }
    return (i < 0 || i >= n) ? -1 : i;
}

template <class R>
struct V3 {
    R x, y, z;
};
using D3 = V3<double>;
template <class R>
__device__ __forceinline__ V3<R> ld3(const R* p) { return {p[0], p[1], p[2]}; }
// a vertex in FP64 (geometry reductions, ray tracing)
template <class R>
__device__ __forceinline__ D3 ld3d(const R* p) { return {(double)p[0], (double)p[1], (double)p[2]}; }
template <class R>
__device__ __forceinline__ V3<R> operator-(V3<R> a, V3<R> b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
template <class R>
__device__ __forceinline__ V3<R> operator+(V3<R> a, V3<R> b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
template <class R>
__device__ __forceinline__ V3<R> operator*(R s, V3<R> a) { return {s * a.x, s * a.y, s * a.z}; }
template <class R>
__device__ __forceinline__ V3<R> operator/(V3<R> a, R s) { return {a.x / s, a.y / s, a.z / s}; }
template <class R>
__device__ __forceinline__ R dot(V3<R> a, V3<R> b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
template <class R>
__device__ __forceinline__ V3<R> cross(V3<R> a, V3<R> b)
{
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
template <class R>
__device__ __forceinline__ R norm(V3<R> a) { return sqrt(dot(a, a)); }
template <class R>
__device__ __forceinline__ void st3(R* p, V3<R> a) { p[0] = a.x; p[1] = a.y; p[2] = a.z; }

struct Grid {
    int n[3];
    int per[3];
    int nt[3];
};

Grid grid_of(const bl_lattice_s* L)
{
    Grid g;
    g.n[0] = L->nx; g.n[1] = L->ny; g.n[2] = L->nz;
    for (int d = 0; d < 3; ++d) g.per[d] = L->periodic[d];
    g.nt[0] = L->ntx; g.nt[1] = L->nty; g.nt[2] = L->ntz;
    return g;
}

// Workgroup order of the immersed-boundary launches over the XCDs: chunks
// of 2^lc consecutive workgroups on one XCD, so that neighbouring vertices
// (which share stencil nodes, element records and tiles) meet in one L2;
// lc = 0 is the hardware's order.  Every order gives the same values.
__device__ __forceinline__ long ibm_block(long bx, long nbx, int lc)
{
    return lc > 0 ? (long)xcd_chunk_block((unsigned)bx, (unsigned)nbx, (unsigned)lc) : bx;
}

// ------------------------------------------------------------- binning
// Stencil bases are stored wrapped into [0, n) on periodic axes (raw on the
// others), so node k of a stencil is base + k minus n at most once.
__device__ __forceinline__ int node_at(int bw, int k, int n, int per)
{
    int v = bw + k;
    if (per) return v >= n ? v - n : v;
    return (v < 0 || v >= n) ? -1 : v;
}

// Distinct tiles touched along one axis by the S (<= 4) nodes of a stencil:
// at most 3 (two for the run up to the face, one more after a periodic
// wrap), kept in registers.
struct AxisTiles {
    int t0 = -1, t1 = -1, t2 = -1, m = 0;
    // by masks: as a choice of fields they became indexed loads from scratch
    __device__ __forceinline__ int get2(int i) const { return t0 ^ ((t0 ^ t1) & -i); }  // i 0 or 1
    __device__ __forceinline__ int get(int i) const
    {
        return t0 ^ ((t0 ^ t1) & -(int)(i == 1)) ^ ((t0 ^ t2) & -(int)(i == 2));
    }
};

__device__ __forceinline__ AxisTiles axis_tiles(int bw, int S, int n, int per)
{
    AxisTiles r;
    if (bw >= 0 && bw + S <= n) {  // nearly every stencil: no face inside it
        r.t0 = bw >> 2;
        r.t1 = (bw + S - 1) >> 2;
        r.m = r.t1 != r.t0 ? 2 : 1;
        return r;
    }
#pragma unroll 1
    for (int k = 0; k < S; ++k) {
        const int node = node_at(bw, k, n, per);
        const int t = node >> 2;
        const bool fresh = node >= 0 && t != r.t0 && t != r.t1 && t != r.t2;
        if (fresh) {
            if (r.m == 0) r.t0 = t;
            else if (r.m == 1) r.t1 = t;
            else r.t2 = t;
            ++r.m;
        }
    }
    return r;
}

// First node of a stencil of half support h (unwrapped), and the same
// wrapped on a periodic axis (node_at's base).
template <class R>
__device__ __forceinline__ int stencil_first(R x, R h) { return (int)ceil(x - h); }

__device__ __forceinline__ int stencil_base(int first, int n, int per)
{
    if (!per || (first >= 0 && first < n)) return first;
    const int b = first % n;
    return b < 0 ? b + n : b;
}

// The stencil's weights along one axis, of the nodes first .. first + 3
// (zero past the support).  The nodes' distances are r + 1, r, 1 - r, 2 - r
// (Peskin) and 1 + r, r, 1 - r (Roma) with r = x - (first + 1), and phi's
// square roots at all of them are the one at r: 1 + 4 r (1 - r) and
// 1 - 3 r^2.  In registers by name: an indexed array here went to scratch.
// The kernel is the stencil's width SW (Peskin 4, Roma 3, top hat 2) at
// compile time: of a run-time choice among the three the compiler made code
// that left the top hat's first weight unset.
template <class R>
struct W4 {
    R w0, w1, w2, w3;
};

__host__ __device__ constexpr int kernel_of(int SW)
{
    return SW == 4 ? BL_KERNEL_PESKIN : (SW == 3 ? BL_KERNEL_ROMA : BL_KERNEL_TOPHAT);
}

template <int SW, class R>
__device__ __forceinline__ W4<R> axis_weights(R x, int first)
{
    constexpr int kernel = kernel_of(SW);
    const R r = x - (R)(first + 1);
    if (kernel == BL_KERNEL_PESKIN) {
        const R q = sqrt(R(1) + R(4) * r * (R(1) - r));
        const R a = R(3) - R(2) * r, b = R(1) + R(2) * r;
        return {R(0.125) * (a - q), R(0.125) * (a + q), R(0.125) * (b + q), R(0.125) * (b - q)};
    }
    if (kernel == BL_KERNEL_ROMA) {
        const R q = sqrt(R(1) - R(3) * r * r);
        constexpr R s = R(1.0) / R(6.0);
        return {s * (R(2) - R(3) * r - q), (R(1.0) / R(3.0)) * (R(1) + q), s * (R(2) + R(3) * r - q), R(0)};
    }
    return {-r, R(1) + r, R(0), R(0)};
}

// The weights on four consecutive nodes, `shift` nodes past the stencil's
// first one (-3 .. 3; zero where the stencil does not reach): three
// conditional shifts by 4, 2 and 1.
template <class R>
__device__ __forceinline__ void shifted(const W4<R>& w, int shift, R o[4])
{
    const int t = shift + 3;
    const bool b4 = t & 4, b2 = t & 2, b1 = t & 1;
    const R z = R(0);
    const R y0 = b4 ? w.w1 : z, y1 = b4 ? w.w2 : z, y2 = b4 ? w.w3 : z, y3 = b4 ? z : w.w0, y4 = b4 ? z : w.w1,
            y5 = b4 ? z : w.w2, y6 = b4 ? z : w.w3;
    const R z0 = b2 ? y2 : y0, z1 = b2 ? y3 : y1, z2 = b2 ? y4 : y2, z3 = b2 ? y5 : y3, z4 = b2 ? y6 : y4;
    o[0] = b1 ? z1 : z0;
    o[1] = b1 ? z2 : z1;
    o[2] = b1 ? z3 : z2;
    o[3] = b1 ? z4 : z3;
}

// Tiles touched by a vertex's stencil: the product of the per-axis sets.
struct StencilTiles {
    AxisTiles ax[3];
    template <class R>
    __device__ __forceinline__ void init(const Grid& gd, int S, R h, const R x[3])
    {
#pragma unroll
        for (int a = 0; a < 3; ++a)
            ax[a] = axis_tiles(stencil_base(stencil_first(x[a], h), gd.n[a], gd.per[a]), S, gd.n[a], gd.per[a]);
    }
    // tile (i, j, k) of the product, or -1 past the per-axis counts
    __device__ __forceinline__ int at(const Grid& gd, int i, int j, int k) const
    {
        if (i >= ax[0].m || j >= ax[1].m || k >= ax[2].m) return -1;
        return (ax[0].get(i) * gd.nt[1] + ax[1].get(j)) * gd.nt[2] + ax[2].get(k);
    }
    // the same for i, j, k of 0 or 1
    __device__ __forceinline__ int at2(const Grid& gd, int i, int j, int k) const
    {
        if (i >= ax[0].m || j >= ax[1].m || k >= ax[2].m) return -1;
        return (ax[0].get2(i) * gd.nt[1] + ax[1].get2(j)) * gd.nt[2] + ax[2].get2(k);
    }
    __device__ __forceinline__ bool wide() const { return ax[0].m > 2 || ax[1].m > 2 || ax[2].m > 2; }
};

// Neighbouring vertices of a membrane touch the same few tiles, so a
// workgroup first aggregates its (tile, vertex) pairs in an LDS hash table
// (open addressing, linear probing) and then issues one global atomic per
// distinct tile.  A pair whose tile finds no slot within kProbes goes
// straight to the global counter; counts stay exact either way.  A workgroup
// of one vertex per lane group has at most 256 tiles (twice that near a
// wall) and 2^9 slots.  One of eight, 256 neighbouring vertices, touches a
// few dozen to some hundred, but 256 scattered over a large membrane up to
// 2 048: 2^10 slots (132 x 111 x 124 suspension, FP64, 71 184 vertices in
// meshes of 642 and 2 562: 282 us a coupled step with 2^9, 274), and no
// more probes, which there are spent for nothing (one membrane of 40 962
// vertices, FP32, 2^9 slots, in the many form: 363 us with 512 probes, 164
// with 16; timed again, in a longer step, 217 with 64, 186 with 16).
constexpr int kProbes = 16;

template <int BITS>
__device__ __forceinline__ int hash_insert(int* keys, int t)
{
    unsigned h = ((unsigned)t * 2654435761u) >> (32 - BITS);
#pragma unroll 1
    for (int probe = 0; probe < kProbes; ++probe) {
        const int old = atomicCAS(&keys[h], -1, t);
        if (old == -1 || old == t) return (int)h;
        h = (h + 1) & ((1 << BITS) - 1);
    }
    return -1;
}

// Readies list `act` (length *na) / flag buffer `flags` for a binning:
// clears the flags of the tiles the list held (two steps back), then the
// last workgroup to finish empties the list and its pair count.  The first
// kResetBlocks workgroups of the grid that carries it take part (all their
// threads); they have read the length before they arrive, so no fence is
// needed, and a bounded number of them keeps the arrival atomic cheap.
constexpr int kResetBlocks = 256;
struct ListReset {
    const int* act = nullptr;  // null: nothing to reset
    int* na = nullptr;
    unsigned char* flags = nullptr;
    int* pairs = nullptr;
    int* arrive = nullptr;
    int* nbig = nullptr;
};

__device__ __forceinline__ void list_reset(const ListReset& lr, int bx, int nbx)
{
    const int nb = min(nbx, kResetBlocks);
    if (bx >= nb) return;
    __shared__ int n;
    if (threadIdx.x == 0) n = *lr.na;
    __syncthreads();
    for (int i = bx * blockDim.x + threadIdx.x; i < n; i += nb * blockDim.x) lr.flags[lr.act[i]] = 0;
    __syncthreads();
    if (threadIdx.x == 0) {
        if (atomicAdd(lr.arrive, 1) == nb - 1) {
            *lr.na = 0;
            *lr.pairs = 0;
            *lr.nbig = 0;
            *lr.arrive = 0;
        }
    }
}

__global__ void __launch_bounds__(256) k_bin_prep(ListReset lr) { list_reset(lr, blockIdx.x, gridDim.x); }

// Near-wall vertices (a boundary is set and the vertex is nearer to it than
// the kernel's half support + 1, src/fsi/ImmersedBoundaryDynamics.hh:
// 346-357) spread after every other vertex, the kernel part (force scaled by
// the blend weight w) before the top-hat part (force scaled by 1 - w), as
// src/fsi/ImmersedBoundaryDynamics_forces.hh:193-237,259-277 orders them.
// List entries carry that order in their value: v for a bulk vertex,
// kNearKey | 2v for the kernel part and kNearKey | 2v + 1 for the top-hat
// part of a near-wall vertex, so sorting a tile's entries gives the
// reference's summation order.
constexpr int kNearKey = 1 << 30;

template <class R>
struct NearView {
    bl_boundary b;
    int on = 0;                      // a boundary is set
    unsigned char* near = nullptr;   // per vertex: near-wall
    R* blend = nullptr;              // per vertex: distance - half support
};

// The first pair that reaches a tile (outside a workgroup's table) lists it
// as touched and flags it as carrying spread force.
__device__ __forceinline__ void touch_tile(int t, int* act, int* na, unsigned char* flags)
{
    act[atomicAdd(na, 1)] = t;
    flags[t] = 1;
}

// Binning in one pass: the tiles each vertex's stencil touches, and every
// (tile, vertex) pair written into the tile's fixed-capacity list (entry
// values as described at kNearKey; a near-wall vertex also gets its blend
// weight and the tiles of its top-hat stencil).  The vertex's position is
// copied to `vp` (x, y, z, 1; all zero for a vertex that takes no part):
// spreading and interpolation form the stencil weights from that copy, one
// aligned load, while the advection moves the vertex itself.  Eight lanes
// take a vertex, one per tile of the 2 x 2 x 2 product.  Per workgroup the
// pairs are counted per distinct tile in LDS (the count at its insert is a
// pair's place in the workgroup's run), one global atomic per tile reserves
// the run.  The order within a list is whatever the atomics give; spreading
// sorts.  The add that takes a tile past BinArgs::small entries appends it
// to the big-tile list.
// Bound by latency on one cell and by instructions on many.  A thread per
// vertex walking its tiles twice, with the weights stored (60 B a vertex in
// FP32), took 16 us beside the element forces for 642 vertices and 99 us for
// 400 800; this takes 7.1 and 87 us.
// Vertices per lane group: one, and kBinMany from kManyVertices on, where
// the chip is full and a workgroup of 256 vertices has fewer distinct tiles
// per pair, so fewer global atomics.  Coupled steps, FP32, one | many: 10 272
// vertices of 642-vertex cells 167 | 170 us, 20 544 188 | 188, 30 816 207 |
// 201, 61 632 252 | 226; 46 224 in FP64 174 | 156.  A subdivided
// sphere's numbering scatters the more the larger it is, so meshes above
// kMeshVertices on average wait until kManyAny: one of 40 962 159 | 164, two
// 284 | 271, eight of 10 242 376 | 350 (these three with 2^9 slots).  No
// mesh between 10 242 and 40 962 was timed; the line lies in that gap.
constexpr int kBinLanes = 8;
constexpr long kManyVertices = 24576, kManyAny = 65536, kMeshVertices = 16384;
constexpr int kBinMany = 8;

template <class R>
struct BinArgs {
    Grid gd;
    int S;
    double h;
    long NV;
    const R* pos;
    Vel4<R>* vp;
    int *count, *list;
    int cap;
    int *act, *na;
    unsigned char* flags;
    int *status, *pairs, *big, *nbig;
    int small;  // entries past which a tile joins the big-tile list
    NearView<R> nw;
    int xcd;  // workgroup order (ibm_block)
};

// One pair past the workgroup's table, straight into the tile's list.
template <class R>
__device__ __forceinline__ void put_pair(const BinArgs<R>& A, int t, int entry, int* n_pairs)
{
    const int slot = atomicAdd(&A.count[t], 1);
    if (slot == 0) touch_tile(t, A.act, A.na, A.flags);
    if (slot == A.small) A.big[atomicAdd(A.nbig, 1)] = t;
    atomicAdd(n_pairs, 1);
    if (slot >= A.cap) atomicOr(&A.status[2], 1);
    else A.list[(long)t * A.cap + slot] = entry;
}

// This lane's tile of a stencil counted in the table: slot and rank there
// (slot * 65536 + rank), or -1 when there is nothing left to place.
template <int BITS, class R>
__device__ __forceinline__ int count_pair(const BinArgs<R>& A, const StencilTiles& st, int r, int entry, int* keys,
                                          int* cnt, int* n_pairs)
{
    // tiles past the 2 x 2 x 2 product: a third one on an axis (a wrap at a
    // size that is no multiple of 4), and a full table
    int direct = -1;
    const int t = st.at2(A.gd, r >> 2, (r >> 1) & 1, r & 1);
    int code = -1;
    if (t >= 0) {
        const int sl = hash_insert<BITS>(keys, t);
        if (sl >= 0) code = (sl << 16) + atomicAdd(&cnt[sl], 1);
        else direct = t;
    }
    if (direct >= 0 || st.wide()) {
#pragma unroll 1
        for (int q = r - kBinLanes; q < 27; q += kBinLanes) {
            const int i = q / 9, j = q / 3 % 3, k = q % 3;
            int tq = direct;
            direct = -1;
            if (q >= 0) tq = i == 2 || j == 2 || k == 2 ? st.at(A.gd, i, j, k) : -1;
            if (tq >= 0) put_pair(A, tq, entry, n_pairs);
        }
    }
    return code;
}

template <class R>
__device__ __forceinline__ void place_pair(const BinArgs<R>& A, int code, int entry, const int* keys, const int* cnt)
{
    if (code < 0) return;
    const int sl = code >> 16, slot = cnt[sl] + (code & 0xffff);
    if (slot < A.cap) A.list[(long)keys[sl] * A.cap + slot] = entry;
}

// ITER vertices per group of lanes, NEAR: a boundary is set (a near-wall
// vertex's code carries kNearCode, and its top-hat entry takes a second one).
constexpr int kNearCode = 1 << 30;

template <class R, bool NEAR, int ITER>
__device__ __forceinline__ void bin_body(long bx, const BinArgs<R>& A)
{
    constexpr int kBits = ITER > 1 ? 10 : 9, kHash = 1 << kBits;
    __shared__ int keys[kHash];
    __shared__ int cnt[kHash];    // pairs per slot, then the run's first index in the tile's list
    __shared__ int fresh[kHash];  // tiles this workgroup reached first
    __shared__ int occ[kHash];    // occupied slots, compacted
    __shared__ int codes[ITER > 1 ? (NEAR ? 2 : 1) * ITER * 256 : 1];
    __shared__ int n_fresh, n_pairs, fresh_base, n_occ;
    for (int i = threadIdx.x; i < kHash; i += blockDim.x) {
        keys[i] = -1;
        cnt[i] = 0;
    }
    if (threadIdx.x == 0) {
        n_fresh = 0;
        n_pairs = 0;
        n_occ = 0;
    }
    const int r = threadIdx.x & (kBinLanes - 1);
    const int vpw = blockDim.x / kBinLanes;
    const long v0 = bx * vpw * ITER + threadIdx.x / kBinLanes;
    const NearView<R>& nw = A.nw;
    const R* __restrict__ pos = A.pos;
    int code = -1, codet = -1, e0 = -1, e1 = -1;
    // the next vertex's position loads while this one is binned
    R nx[3];
    for (int a = 0; a < 3; ++a) nx[a] = pos[3 * min(v0, A.NV - 1) + a];
    __syncthreads();
#pragma unroll 1
    for (int it = 0; it < ITER; ++it) {
        const long v = v0 + it * vpw;
        const R x[3] = {nx[0], nx[1], nx[2]};
        if (it + 1 < ITER) {
            const long vn = min(v + vpw, A.NV - 1);
            for (int a = 0; a < 3; ++a) nx[a] = pos[3 * vn + a];
        }
        code = codet = e0 = -1;
        if (v < A.NV) {
            // a vertex whose position is not finite (a membrane that blew
            // up) or absurdly far off touches no tile and is reported
            const bool off = !(fabs(x[0]) < R(1e9)) || !(fabs(x[1]) < R(1e9)) || !(fabs(x[2]) < R(1e9));
            if (r == 0) {
                A.vp[v] = off ? Vel4<R>{R(0), R(0), R(0), R(0)} : Vel4<R>{x[0], x[1], x[2], R(1)};
                if (off) atomicOr(&A.status[2], 4);
            }
            if (!off) e0 = (int)v;
            if (NEAR) {
                // the wall distance in FP64 (the boundary's own arithmetic)
                const double p[3] = {(double)x[0], (double)x[1], (double)x[2]};
                const bool nr = !off && bnd_less_than(nw.b, p, A.h + 1.);
                const R wb = off ? R(1.0) : (R)(bnd_distance(nw.b, p) - A.h);
                if (r == 0) {
                    nw.near[v] = nr;
                    nw.blend[v] = wb;
                }
                if (nr) {
                    e0 = wb > R(0) ? (kNearKey | (int)(2 * v)) : -1;
                    if (wb < R(1)) {
                        e1 = kNearKey | (int)(2 * v + 1);
                        StencilTiles stt;
                        stt.init(A.gd, 2, R(1.0), x);
                        codet = count_pair<kBits>(A, stt, r, e1, keys, cnt, &n_pairs);
                    }
                }
            }
            if (e0 >= 0) {
                StencilTiles st;
                st.init(A.gd, A.S, (R)A.h, x);
                code = count_pair<kBits>(A, st, r, e0, keys, cnt, &n_pairs);
            }
        }
        if (ITER > 1) {
            codes[it * blockDim.x + threadIdx.x] = code >= 0 && (e0 & kNearKey) ? code | kNearCode : code;
            if (NEAR) codes[(ITER + it) * blockDim.x + threadIdx.x] = codet;
        }
    }
    __syncthreads();
    // one global atomic per distinct tile; the occupied slots are compacted
    // first so that each lane waits for one atomic, not one per slot it scans
    for (int i = threadIdx.x; i < kHash; i += blockDim.x)
        if (cnt[i] > 0) occ[atomicAdd(&n_occ, 1)] = i;
    __syncthreads();
    for (int k = threadIdx.x; k < n_occ; k += blockDim.x) {
        const int i = occ[k];
        const int c = cnt[i];
        const int t = keys[i];
        const int old = atomicAdd(&A.count[t], c);
        cnt[i] = old;
        if (old == 0) fresh[atomicAdd(&n_fresh, 1)] = t;
        if (old <= A.small && old + c > A.small) A.big[atomicAdd(A.nbig, 1)] = t;
        atomicAdd(&n_pairs, c);
        if (old + c > A.cap) atomicOr(&A.status[2], 1);
    }
    __syncthreads();
    // the touched-list reservation is issued before the list fill and its
    // result read after it, so the two round trips overlap
    int fb = 0;
    if (threadIdx.x == 0) {
        if (n_fresh) fb = atomicAdd(A.na, n_fresh);
        if (n_pairs) atomicAdd(A.pairs, n_pairs);
    }
    if (ITER > 1) {
#pragma unroll 4
        for (int it = 0; it < ITER; ++it) {
            const int v = (int)(v0 + it * vpw), c = codes[it * blockDim.x + threadIdx.x];
            const bool nr = NEAR && c >= 0 && (c & kNearCode) != 0;
            place_pair(A, nr ? c & ~kNearCode : c, nr ? kNearKey | (2 * v) : v, keys, cnt);
            if (NEAR) place_pair(A, codes[(ITER + it) * blockDim.x + threadIdx.x], kNearKey | (2 * v + 1), keys, cnt);
        }
    } else {
        place_pair(A, code, e0, keys, cnt);
        if (NEAR) place_pair(A, codet, e1, keys, cnt);
    }
    if (threadIdx.x == 0) fresh_base = fb;
    __syncthreads();
    for (int i = threadIdx.x; i < n_fresh; i += blockDim.x) {
        A.act[fresh_base + i] = fresh[i];
        A.flags[fresh[i]] = 1;
    }
}

// A binning workgroup: one vertex per lane group, or kBinMany.  MANY has its
// two forms in kernels of their own: one kernel would hold the LDS of both
// (400 800 vertices, FP32: 82 us alone, 125 together).
enum BinForm { BIN_ONE, BIN_MANY, BIN_MANY_NEAR };

template <class R, BinForm FORM>
__device__ __forceinline__ void bin_group(long bx, const BinArgs<R>& A)
{
    if (FORM == BIN_MANY_NEAR) bin_body<R, true, kBinMany>(bx, A);
    else if (FORM == BIN_MANY) bin_body<R, false, kBinMany>(bx, A);
    else if (A.nw.on) bin_body<R, true, 1>(bx, A);
    else bin_body<R, false, 1>(bx, A);
}

template <class R, BinForm FORM>
__global__ void __launch_bounds__(256) k_bin(BinArgs<R> a)
{
    bin_group<R, FORM>(ibm_block(blockIdx.x, gridDim.x, a.xcd), a);
}

__global__ void k_clear_bins(int* count, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) count[i] = 0;
}

__global__ void k_zero_u8(unsigned char* p, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void k_fill_i32(int* p, long n, int v)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}


// ------------------------------------------------------------ membrane
template <class R>
struct ForceView {
    int np;
    const long *p_voff, *p_toff, *p_loff, *p_poff;
    const int *p_shape, *p_model, *p_bug;
    const double* p_params;
    const double* p_geom;
    const int *s_voff, *s_toff, *s_loff, *s_poff, *s_vtoff, *s_vloff, *s_vpoff;
    const int* s_tri;
    const double *s_tri_area0, *s_tri_geo0;
    const int* s_link;
    const double* s_link_len;
    const int* s_pair;
    const double* s_pair_cs0;
    const int *s_vt_head, *s_vt, *s_vl_head, *s_vl, *s_vp_head, *s_vp;
    const double* s_area0;
    const R* pos;
    const int *v_part, *t_part, *r_part, *l_part;  // particle of each vertex / triangle / pair / link
    const int4* v_inc;  // per vertex: {link list start, links, triangle list start, triangles},
                        // {pair list start, pairs, particle, 0}; counts of unused kinds are 0
};

// Element forces are bound by the vector units: a suspension of 400 cells
// (FP32) took 87 us when every quotient of the formulas was a division (67 of
// them, about 12 instructions each) and takes 56.  So lengths are inverted
// once, the three vertices share their scalar factors, and a force that is
// minus the sum of the others is formed as that.  Errors of a cell's forces,
// meshes of 162 to 2 562 vertices, against before: FP64 against long double
// 0.87 to 0.99 (in-plane alone), 0.91 to 1.18 with the constraints, whose
// error is that of the volume's sum; FP32 against FP64 0.85 to 1.01.

// Skalak / NeoHookean in-plane forces of one triangle
// (src/fsi/DeformableCapsule.hh:60-150), with the reference's
// c = l' sin(phi) / (l' sin(phi0)) when `bug` is set.  The energy's gradient
// w1 grad I1 + w2 grad I2 is collected into the factors of the gradients of
// l, l' and cos(phi), whose vectors are multiples of the two edges; w1 + w2
// vanishes at rest and is taken without the cancellation.
template <class R>
__device__ void capsule_triangle(V3<R> p0, V3<R> p1, V3<R> p2, const double* geo0, double area0_, double G_,
                                 double Cc_, bool skalak, bool bug, V3<R> out[3])
{
    using V = V3<R>;
    const R area0 = (R)area0_, G = (R)G_, Cc = (R)Cc_;
    const V e0 = p1 - p0, e1 = p2 - p0;
    const R l = norm(e0), lp = norm(e1);
    const R cos_phi0 = (R)geo0[2], sin_phi0 = (R)geo0[3];
    const R l0 = (R)geo0[0], l0p = (R)geo0[1];
    const R il = R(1) / l, ilp = R(1) / lp, il0 = R(1) / l0, il0p = R(1) / l0p, is0 = R(1) / sin_phi0;
    const R d = dot(e0, e1), n = norm(cross(e0, e1));
    // a, b and c lose digits in the strains below: their quotients are divisions
    const R a = l / l0, ap = lp * il0p, q = R(1) / (l * l0p);
    const R b = (d * q - a * cos_phi0) / sin_phi0;
    const R c = (bug ? n / (l * lp) : n * q) / sin_phi0;
    const R cos_phi = d * il * ilp;
    const R D11 = (a * a - R(1)) * R(0.5);
    const R D22 = (b * b + c * c - R(1)) * R(0.5);
    const R D12 = a * b * R(0.5);
    const R I1 = R(2) * (D11 + D22);
    const R I2 = I1 + R(4) * (D11 * D22 - D12 * D12);
    R w2, w12;  // w2 and w1 + w2
    if (skalak) {
        w2 = Cc * I2 - R(1);
        w12 = I1 + Cc * I2;
    } else {
        const R i = R(1) / (R(1) + I2);
        w2 = -i * i;
        w12 = I2 * (R(2) + I2) * (i * i);
    }
    const R k = -R(0.5) * G * area0;
    const R s11 = k * (R(2) * w12 + R(4) * w2 * D22);
    const R s22 = k * (R(2) * w12 + R(4) * w2 * D11) * (is0 * is0);
    const R s12 = -R(4) * k * w2 * D12 * (il0p * is0);
    const R r = il0 * cos_phi0, t = il0p * cos_phi;
    const R cl = s11 * a * il0 + s22 * (l * r - lp * t) * r + s12 * (lp * t - R(2) * l * r);
    const R clp = s22 * (ap - l * r * cos_phi) * il0p + s12 * l * t;
    const R x = il0p * (s12 - s22 * r);
    const V f1 = (il * (cl - x * lp * cos_phi)) * e0 + x * e1;
    const V f2 = x * e0 + (ilp * (clp - x * l * cos_phi)) * e1;
    out[0] = V{R(0), R(0), R(0)} - (f1 + f2);
    out[1] = f1;
    out[2] = f2;
}

// Area (local + global) and volume constraint forces of one triangle
// (src/fsi/RBCParticle.hh:176-209, src/fsi/TriangleUtils.h:60-129).
template <class R>
__device__ void area_volume_triangle(V3<R> v0, V3<R> v1, V3<R> v2, double area0_, double A0tot_, double A_, double V_,
                                     double k_ag_, double k_al_, double k_v_, double V0_, V3<R> out[3])
{
    const R area0 = (R)area0_, A0tot = (R)A0tot_, A = (R)A_, V = (R)V_, k_ag = (R)k_ag_, k_al = (R)k_al_,
            k_v = (R)k_v_, V0 = (R)V0_;
    const V3<R> n = cross(v0 - v1, v0 - v2);
    const R la2 = norm(n);  // twice the area
    const R df_area = (k_ag * (A0tot - A) / A0tot + k_al * (area0 - R(0.5) * la2) / area0) * (R(0.5) / la2);
    const R df_vol = k_v * (V0 - V) / (R(6.) * V0);
    const V3<R> m = df_area * n;
    const V3<R> g1 = cross(m, v0 - v2), g2 = cross(m, v1 - v0);
    out[0] = (out[0] - (g1 + g2)) + df_vol * cross(v1, v2);
    out[1] = (out[1] + g1) + df_vol * cross(v2, v0);
    out[2] = (out[2] + g2) + df_vol * cross(v0, v1);
}

// Force of one link on its first vertex (the second gets the negative):
// worm-like chain + power-law repulsion (src/fsi/RBCParticle.hh:149-171,
// exponent 2).  The link's coefficients depend on the rest length l0 and the
// modulus G only: with k1 and k2 the two derivatives of the chain's energy
// at rest, ks = (4 G / sqrt 3) l0 / (3 k1 + k2) and kp = k1 l0^2 ks.
template <class R>
__device__ V3<R> link_force(const ForceView<R>& f, int s, long vo, const double* P, long link)
{
    constexpr double x0 = 1. / 2.2, y0 = 1 - x0;
    constexpr double k1 = 0.25 * (6. * x0 + (3 * x0 * x0 - 2 * x0 * x0 * x0) / (y0 * y0));
    constexpr double k2 = x0 / (2. * y0 * y0 * y0) + 0.25 * (1. - 1. / (y0 * y0));
    constexpr double kInvSqrt3 = 0.57735026918962576451;
    const long sl = f.s_loff[s] + link;
    const double l0d = f.s_link_len[sl];
    const double ksd = (4. * kInvSqrt3 / (3. * k1 + k2)) * l0d * P[0];
    const R ks = (R)ksd;
    const R kp = (R)(k1 * l0d * l0d * ksd);
    const int2 q = ((const int2*)f.s_link)[sl];
    const V3<R> dv = ld3(f.pos + 3 * (vo + q.x)) - ld3(f.pos + 3 * (vo + q.y));
    const R L = norm(dv);
    const R x = L / ((R)l0d * R(2.2)), y = R(1) - x;
    const R df = -R(0.25) * ks * (R(6.) * x + (R(3.) - R(2.) * x) * (x * x) / (y * y)) + kp / (L * L);
    return (df / L) * dv;
}

// Forces of one triangle on its three vertices.
template <class R>
__device__ void tri_forces(const ForceView<R>& f, int p, int s, int model, long vo, const double* P, long tri,
                           V3<R> out[3])
{
    const long st = f.s_toff[s] + tri;
    const int i0 = f.s_tri[3 * st], i1 = f.s_tri[3 * st + 1], i2 = f.s_tri[3 * st + 2];
    const V3<R> v0 = ld3(f.pos + 3 * (vo + i0)), v1 = ld3(f.pos + 3 * (vo + i1)), v2 = ld3(f.pos + 3 * (vo + i2));
    out[0] = out[1] = out[2] = V3<R>{R(0), R(0), R(0)};
    const double area0 = f.s_tri_area0[st];
    if (model == BL_MODEL_CAPSULE_SKALAK || model == BL_MODEL_CAPSULE_NEOHOOKEAN || model == 3)
        capsule_triangle<R>(v0, v1, v2, f.s_tri_geo0 + 4 * st, area0, P[0], P[1],
                            model != BL_MODEL_CAPSULE_NEOHOOKEAN, f.p_bug[p] != 0, out);
    if (model == BL_MODEL_RBC || model == 3)
        area_volume_triangle<R>(v0, v1, v2, area0, f.s_area0[s], f.p_geom[kGeomSums * p], f.p_geom[kGeomSums * p + 1], P[2], P[3],
                                P[4], P[5], out);
}

// Bending forces of one dihedral pair on its four vertices.
template <class R>
__device__ void pair_forces(const ForceView<R>& f, int s, long vo, const double* P, long pair, V3<R> out[4])
{
    using V = V3<R>;
    const long sp = f.s_poff[s] + pair;
    const int4 q = ((const int4*)f.s_pair)[sp];
    const V v0 = ld3(f.pos + 3 * (vo + q.x)), v1 = ld3(f.pos + 3 * (vo + q.y));
    const V v2 = ld3(f.pos + 3 * (vo + q.z)), v3 = ld3(f.pos + 3 * (vo + q.w));
    const V e0 = v1 - v0, e1 = v2 - v0, e2 = v3 - v0;
    const R e1n = norm(e1), ie = R(1) / e1n;
    const V n1 = cross(e0, e1), n2 = cross(e1, e2);
    const R i1 = R(1) / norm(n1), i2 = R(1) / norm(n2);
    // sine and cosine of the angle, times both normals' lengths
    const R cs = dot(n1, n2);
    const R sn = ((dot(n1 - n2, v1 - v3) > R(0)) ? R(1.0) : -R(1.0)) * norm(cross(n1, n2));
    const R pref = (R)P[6] * (-(R)f.s_pair_cs0[2 * sp] * sn + (R)f.s_pair_cs0[2 * sp + 1] * cs) * (i1 * i2);
    const V a1 = (pref * i1 * i1) * n1, a2 = (pref * i2 * i2) * n2;
    out[0] = (dot(e1, e1 - e2) * ie) * a2 + (dot(e1, e1 - e0) * ie) * a1;
    out[1] = -e1n * a1;
    out[2] = (dot(e1, e2) * ie) * a2 + (dot(e1, e0) * ie) * a1;
    out[3] = -e1n * a2;
}

// One thread per element, over the concatenation [triangles | pairs | links]
// of all particles: the element's forces on its vertices go to its own slots
// of `ec` (9 values per triangle, 12 per pair, 3 per link).  Elements that
// the particle's model does not use are skipped.
template <class R>
struct ElemArgs {
    ForceView<R> f;
    long NT, NP, NL, ec_pair, ec_link;
    R* ec;
    int xcd;  // workgroup order (ibm_block)
};

template <class R>
__device__ __forceinline__ void elem_body(long bx, const ElemArgs<R>& A)
{
    const ForceView<R>& f = A.f;
    const long NT = A.NT, NP = A.NP, NL = A.NL, ec_pair = A.ec_pair, ec_link = A.ec_link;
    R* __restrict__ ec = A.ec;
    const long e = bx * blockDim.x + threadIdx.x;
    if (e < NT) {
        const int p = f.t_part[e];
        V3<R> out[3];
        tri_forces<R>(f, p, f.p_shape[p], f.p_model[p], f.p_voff[p], f.p_params + 8 * p, e - f.p_toff[p], out);
        for (int k = 0; k < 3; ++k) st3(ec + 9 * e + 3 * k, out[k]);
    } else if (e < NT + NP) {
        const long g = e - NT;
        const int p = f.r_part[g];
        const int model = f.p_model[p];
        if (model != BL_MODEL_RBC && model != 3) return;
        V3<R> out[4];
        pair_forces<R>(f, f.p_shape[p], f.p_voff[p], f.p_params + 8 * p, g - f.p_poff[p], out);
        for (int k = 0; k < 4; ++k) st3(ec + ec_pair + 12 * g + 3 * k, out[k]);
    } else if (e < NT + NP + NL) {
        const long g = e - NT - NP;
        const int p = f.l_part[g];
        if (f.p_model[p] != BL_MODEL_RBC) return;
        st3(ec + ec_link + 3 * g, link_force<R>(f, f.p_shape[p], f.p_voff[p], f.p_params + 8 * p, g - f.p_loff[p]));
    }
}

template <class R>
__global__ void __launch_bounds__(256) k_elem_forces(ElemArgs<R> a)
{
    elem_body<R>(ibm_block(blockIdx.x, gridDim.x, a.xcd), a);
}

// Force on every vertex: the contributions of its incident elements --
// links (src/fsi/RBCParticle.hh:149-171), triangles
// (src/fsi/DeformableCapsule.hh:60-150, src/fsi/RBCParticle.hh:176-209) and
// pairs (src/fsi/RBCParticle.hh:214-246) -- from the per-element buffer.
// The incidence lists hold element * 4 + the vertex's slot in the element.
// Four lanes per vertex: lane l sums entries l, l+4, ... of the vertex's
// list [links | triangles | pairs] in order, then a fixed butterfly adds the
// lanes, so the result does not depend on scheduling.  No atomics.
// Lane 0 starts from the wall-interaction decorators' forces, which the
// reference applies before the membrane forces, and the sum ends with the
// particle-particle forces (`fpp`), which it adds after them
// (src/fsi/ImmersedBoundaryDynamics_forces.hh:293-301).
// GL (2, 4 or 8) lanes per vertex, a launch parameter (bl_ibm_set_launch):
// the lane count fixes the butterfly, so results agree to rounding across
// lane counts and are bitwise repeatable for each.
constexpr int kGatherLanes = 4;  // the default

template <class R>
struct GatherArgs {
    ForceView<R> f;
    long NV, ec_pair, ec_link;
    const R* ec;
    R* force;
    DecoSet deco;
    const R* fpp;
    const R* ext;  // host-given vertex forces, added after the decorators (or null)
    int xcd;       // workgroup order (ibm_block)
};

template <class R, int GL>
__device__ __forceinline__ void gather_body(long bx, const GatherArgs<R>& A)
{
    const ForceView<R>& f = A.f;
    const long NV = A.NV, ec_pair = A.ec_pair, ec_link = A.ec_link;
    const R* __restrict__ ec = A.ec;
    R* __restrict__ force = A.force;
    const DecoSet& deco = A.deco;
    const R* __restrict__ fpp = A.fpp;
    const long gid = bx * blockDim.x + threadIdx.x;
    const long v = gid / GL;
    const int lane = (int)(gid % GL);
    R c0 = R(0), c1 = R(0), c2 = R(0);
    if (deco.n && lane == 0 && v < NV) {
        // the decorators' potentials and wall geometry in FP64
        const double p[3] = {(double)f.pos[3 * v], (double)f.pos[3 * v + 1], (double)f.pos[3 * v + 2]};
        double w[3] = {0, 0, 0};
        deco_apply(deco, p, w);
        c0 = (R)w[0];
        c1 = (R)w[1];
        c2 = (R)w[2];
    }
    if (A.ext && lane == 0 && v < NV) {
        c0 += A.ext[3 * v];
        c1 += A.ext[3 * v + 1];
        c2 += A.ext[3 * v + 2];
    }
    if (v < NV) {
        // the vertex's incidence lists in one load (built at init), so the
        // element forces are two dependent loads away
        const int4 ia = f.v_inc[2 * v], ib = f.v_inc[2 * v + 1];
        const int p = ib.z;
        const int nl = ia.y, nt = ia.w, npr = ib.y;
        const int* Ll = f.s_vl + ia.x;
        const int* Lt = f.s_vt + ia.z;
        const int* Lp = f.s_vp + ib.x;
        const R* El = ec + ec_link + 3 * f.p_loff[p];
        const R* Et = ec + 9 * f.p_toff[p];
        const R* Ep = ec + ec_pair + 12 * f.p_poff[p];
        for (int e = lane; e < nl + nt + npr; e += GL) {
            if (e < nl) {
                const int code = Ll[e];
                const R* x = El + 3 * (code >> 2);
                const R sg = (code & 3) == 0 ? R(1.0) : -R(1.0);
                c0 += sg * x[0];
                c1 += sg * x[1];
                c2 += sg * x[2];
            } else if (e < nl + nt) {
                const int code = Lt[e - nl];
                const R* x = Et + 9 * (code >> 2) + 3 * (code & 3);
                c0 += x[0];
                c1 += x[1];
                c2 += x[2];
            } else {
                const int code = Lp[e - nl - nt];
                const R* x = Ep + 12 * (code >> 2) + 3 * (code & 3);
                c0 += x[0];
                c1 += x[1];
                c2 += x[2];
            }
        }
    }
#pragma unroll
    for (int o = 1; o < GL; o <<= 1) {
        c0 += __shfl_xor(c0, o);
        c1 += __shfl_xor(c1, o);
        c2 += __shfl_xor(c2, o);
    }
    if (lane == 0 && v < NV) {
        if (fpp) {
            c0 += fpp[3 * v];
            c1 += fpp[3 * v + 1];
            c2 += fpp[3 * v + 2];
        }
        force[3 * v] = c0;
        force[3 * v + 1] = c1;
        force[3 * v + 2] = c2;
    }
}

template <class R, int GL>
__global__ void __launch_bounds__(256) k_vertex_gather(GatherArgs<R> a)
{
    gather_body<R, GL>(ibm_block(blockIdx.x, gridDim.x, a.xcd), a);
}

// ------------------------------------------------- velocity staging
// The progs' computeVelocity pass (staged_velocity), restricted to the
// cells of the tiles this step's stencils touch (`touched`, the step's tile
// flags).  `lv` carries the force field and flags of the last collision.
// One thread per cell in z-fastest order, so population reads coalesce as
// in the collide kernel and the staged vectors are written contiguously; or,
// where few tiles of many are touched (stage_by_list), one wave per touched
// tile off the list, since looking at every cell's flag is a launch over the
// whole lattice (384^3 with 2 124 touched tiles: 86 us against 24).
// (With the staging carried by the collision, k_collide_stream writes the
// same values from the populations it loads.)
struct StageArgs {
    LatView lv;
    const unsigned char* touched;
    void* ut;  // Vel4 of the storage's compute type
    const int *active, *nactive;  // the touched-tile list (null: a thread per cell)
    FastDiv dty, dtz;             // division by the tiles along y and z
};

template <class S, bool SWAPPED>
__device__ __forceinline__ void stage_cell(const StageArgs& A, unsigned c, int x, int y, int z)
{
    using C = typename Pop<S>::C;
    using FT = typename Pop<S>::F;
    const LatView& lv = A.lv;
    const unsigned char m = lv.mask ? lv.mask[c] : (unsigned char)M_FLUID;
    // the moments as the collision forms them (working form of the storage),
    // so that a staging carried by the collision gives the same values
    C rb = C(0), j[3] = {C(0), C(0), C(0)};
    if (m == M_FLUID) {
        Nbr nb;
        if (SWAPPED) nb.init(lv, x, y, z);
        C f[Q];
        load_post_w<S>(lv, nb, c, SWAPPED, f);
        wmoments<S>(f, rb, j);
    }
    const C invRho = C(1) / (rb + C(1));
    ((Vel4<C>*)A.ut)[c] = staged_velocity_m<FT, C>(lv, lv.flags, lv.force, m, c, x, y, z, j, invRho);
}

// EITHER: off the touched-tile list where there is one; by cells only
// otherwise.
template <class S, bool SWAPPED, bool EITHER>
__device__ __forceinline__ void stage_body(unsigned bx, unsigned nbx, const StageArgs& A)
{
    const LatView& lv = A.lv;
    if (EITHER && A.active) {
        const int na = *A.nactive, lane = threadIdx.x & 63;
        for (int a = (int)(bx * (blockDim.x >> 6) + (threadIdx.x >> 6)); a < na; a += (int)(nbx * (blockDim.x >> 6))) {
            const unsigned t = (unsigned)A.active[a], r = fdiv(t, A.dtz), tx = fdiv(r, A.dty);
            const int x = (int)tx * kTile + (lane >> 4), y = (int)(r - tx * lv.nty) * kTile + ((lane >> 2) & 3),
                      z = (int)(t - r * lv.ntz) * kTile + (lane & 3);
            if (x < lv.nx && y < lv.ny && z < lv.nz)
                stage_cell<S, SWAPPED>(A, ((unsigned)x * lv.ny + y) * lv.nz + z, x, y, z);
        }
        return;
    }
    const unsigned c = bx * blockDim.x + threadIdx.x;
    if (c >= lv.ncell) return;
    int x, y, z;
    decode(c, lv, x, y, z);
    const unsigned t = ((unsigned)(x >> 2) * lv.nty + (y >> 2)) * lv.ntz + (z >> 2);
    if (A.touched[t]) stage_cell<S, SWAPPED>(A, c, x, y, z);
}

template <class S, bool SWAPPED>
__global__ void __launch_bounds__(256) k_stage_u(StageArgs a) { stage_body<S, SWAPPED, true>(blockIdx.x, gridDim.x, a); }

// ------------------------------------------------------- interpolation
// U_k = sum over the stencil nodes of phi(dx) phi(dy) phi(dz) u
// (src/fsi/ImmersedBoundaryDynamics_interpolation.hh:14-78): a group of
// lanes per vertex, lane (j, k) walks the x-line of its (y, z) node pair
// (nodes outside a non-periodic face skipped, weight (phi_x phi_y) phi_z as
// the reference forms it), then the lanes are added by a fixed butterfly,
// all in FP64.  The lanes of one x-step read consecutive cells of a few
// z-rows.  With MOVE the vertex is then advanced, x += U (explicit Euler,
// src/fsi/DeformableParticle3D.hh:26-36).
// Explicit Euler step that reflects off the boundary
// (DeformableParticle3D::move_vertices, src/fsi/DeformableParticle3D.hh:26-50),
// in FP64 (the boundary's own arithmetic) for either vertex type.
template <class R>
__device__ __forceinline__ void move_reflect(const bl_boundary& b, R* pr, const R* ur)
{
#pragma clang fp contract(off)
    const double u[3] = {(double)ur[0], (double)ur[1], (double)ur[2]};
    const double old[3] = {(double)pr[0], (double)pr[1], (double)pr[2]};
    const double nw[3] = {old[0] + u[0], old[1] + u[1], old[2] + u[2]};
    double t;
    if (!bnd_trace_ray(b, old, nw, t)) {
        pr[0] = (R)nw[0];
        pr[1] = (R)nw[1];
        pr[2] = (R)nw[2];
        return;
    }
    double q[3] = {old[0] + t * u[0], old[1] + t * u[1], old[2] + t * u[2]};
    double n[3];
    bnd_normal(b, q, n);
    const double vn = u[0] * n[0] + u[1] * n[1] + u[2] * n[2];
    for (int a = 0; a < 3; ++a) pr[a] = (R)(q[a] + (u[a] - 2. * vn * n[a]) * (1. - t));
}

// A near-wall vertex (blend weight w < 1) also interpolates with the top
// hat, lanes (j, k) < 2 over its 2x2x2 stencil, and takes (1 - w) u_tophat
// + w u_kernel, or u_tophat alone for w <= 0
// (src/fsi/ImmersedBoundaryDynamics_interpolation.hh:182-230).
template <class R>
struct InterpArgs {
    Grid gd;
    long NV;
    double h;
    const Vel4<R>* vp;  // the binning's position copies
    const void* ut;     // Vel4<C>
    R *vel, *pos;
    ListReset lr;
    NearView<R> nw;
    int xcd;  // workgroup order of the vertices (ibm_block; the list reset keeps the hardware's)
};

template <class C, int SW, bool MOVE, class R>
__device__ __forceinline__ void interp_body(long bx, int nbx, const InterpArgs<R>& A)
{
    const Grid& gd = A.gd;
    const long NV = A.NV;
    const Vel4<C>* __restrict__ ut = (const Vel4<C>*)A.ut;
    R* __restrict__ vel = A.vel;
    R* __restrict__ pos = A.pos;
    const NearView<R>& nw = A.nw;
    if (A.lr.act) list_reset(A.lr, (int)bx, nbx);  // the next binning's list, carried by this launch
    constexpr int kernel = kernel_of(SW);
    constexpr int LA = SW == 2 ? 2 : 4;
    constexpr int LPV = LA * LA;
    const long gid = ibm_block(bx, nbx, A.xcd) * blockDim.x + threadIdx.x;
    const long v = gid / LPV;
    const int r = (int)(gid % LPV);
    const int j = r / LA, k = r % LA;
    R a0 = R(0), a1 = R(0), a2 = R(0);
    const Vel4<R> P = v < NV ? A.vp[v] : Vel4<R>{R(0), R(0), R(0), R(0)};
    const R h = (R)A.h;
    const int fx = stencil_first(P.x, h), fy = stencil_first(P.y, h), fz = stencil_first(P.z, h);
    // the stencil's weights: a lane of the group forms one of the twelve and
    // the group shares them (a top-hat weight costs less than the exchange)
    R wx[SW], wy, wz;
    if (SW == 2) {
#pragma unroll
        for (int i = 0; i < SW; ++i) wx[i] = dirac<R>(kernel, (R)(fx + i) - P.x);
        wy = dirac<R>(kernel, (R)(fy + j) - P.y);
        wz = dirac<R>(kernel, (R)(fz + k) - P.z);
    } else {
        const R mine = dirac<R>(kernel, (j == 0 ? (R)(fx + k) - P.x : (j == 1 ? (R)(fy + k) - P.y : (R)(fz + k) - P.z)));
#pragma unroll
        for (int i = 0; i < SW; ++i) wx[i] = __shfl(mine, i, LPV);
        wy = __shfl(mine, 4 + j, LPV);
        wz = __shfl(mine, 8 + k, LPV);
    }
    if (P.w != R(0) && j < SW && k < SW) {
        const int yj = node_at(stencil_base(fy, gd.n[1], gd.per[1]), j, gd.n[1], gd.per[1]);
        const int zk = node_at(stencil_base(fz, gd.n[2], gd.per[2]), k, gd.n[2], gd.per[2]);
        if (yj >= 0 && zk >= 0) {
            const int b0 = stencil_base(fx, gd.n[0], gd.per[0]);
#pragma unroll
            for (int i = 0; i < SW; ++i) {
                const int xi = node_at(b0, i, gd.n[0], gd.per[0]);
                if (xi < 0) continue;
                const R w = (wx[i] * wy) * wz;
                const Vel4<C> u = ut[((size_t)xi * gd.n[1] + yj) * gd.n[2] + zk];
                a0 += w * (R)u.x;
                a1 += w * (R)u.y;
                a2 += w * (R)u.z;
            }
        }
    }
#pragma unroll
    for (int o = 1; o < LPV; o <<= 1) {
        a0 += __shfl_xor(a0, o);
        a1 += __shfl_xor(a1, o);
        a2 += __shfl_xor(a2, o);
    }
    if (nw.on && v < NV && nw.near[v] && nw.blend[v] < R(1)) {  // the same for all lanes of the vertex
        const R wb = nw.blend[v];
        R t0 = R(0), t1 = R(0), t2 = R(0);
        if (j < 2 && k < 2) {
            const int f[3] = {stencil_first(P.x, R(1.0)), stencil_first(P.y, R(1.0)), stencil_first(P.z, R(1.0))};
            const int yj = node_at(stencil_base(f[1], gd.n[1], gd.per[1]), j, gd.n[1], gd.per[1]);
            const int zk = node_at(stencil_base(f[2], gd.n[2], gd.per[2]), k, gd.n[2], gd.per[2]);
            if (yj >= 0 && zk >= 0) {
                const R ty = dirac<R>(BL_KERNEL_TOPHAT, (R)(f[1] + j) - P.y);
                const R tz = dirac<R>(BL_KERNEL_TOPHAT, (R)(f[2] + k) - P.z);
                for (int i = 0; i < 2; ++i) {
                    const int xi = node_at(stencil_base(f[0], gd.n[0], gd.per[0]), i, gd.n[0], gd.per[0]);
                    if (xi < 0) continue;
                    const R w = (dirac<R>(BL_KERNEL_TOPHAT, (R)(f[0] + i) - P.x) * ty) * tz;
                    const Vel4<C> u = ut[((size_t)xi * gd.n[1] + yj) * gd.n[2] + zk];
                    t0 += w * (R)u.x;
                    t1 += w * (R)u.y;
                    t2 += w * (R)u.z;
                }
            }
        }
#pragma unroll
        for (int o = 1; o < LPV; o <<= 1) {
            t0 += __shfl_xor(t0, o);
            t1 += __shfl_xor(t1, o);
            t2 += __shfl_xor(t2, o);
        }
        if (wb <= R(0)) {
            a0 = t0;
            a1 = t1;
            a2 = t2;
        } else {
            a0 = (R(1.) - wb) * t0 + wb * a0;
            a1 = (R(1.) - wb) * t1 + wb * a1;
            a2 = (R(1.) - wb) * t2 + wb * a2;
        }
    }
    if (r == 0 && v < NV) {
        vel[3 * v] = a0;
        vel[3 * v + 1] = a1;
        vel[3 * v + 2] = a2;
        if (MOVE) {
            if (nw.on) {
                const R u[3] = {a0, a1, a2};
                move_reflect<R>(nw.b, pos + 3 * v, u);
            } else {
                pos[3 * v] += a0;
                pos[3 * v + 1] += a1;
                pos[3 * v + 2] += a2;
            }
        }
    }
}

template <class C, int SW, bool MOVE, class R>
__global__ void __launch_bounds__(256) k_interp(InterpArgs<R> a)
{
    interp_body<C, SW, MOVE, R>(blockIdx.x, gridDim.x, a);
}

// ----------------------------------------------------------- spreading
// Every cell of a touched 4x4x4 tile sums g + phi phi phi F_k over the
// tile's vertices in increasing vertex order, the order of the reference's
// vertex loop (src/fsi/ImmersedBoundaryDynamics_forces.hh:53-85), and writes
// its force.  The tile's list is sorted first.  Then, 64 entries at a time,
// lane e loads entry e and forms its weights on the tile's own 4 cells per
// axis (zero outside the stencil) and its force in registers (all zero past
// the list's end); two halves of 32 go through LDS in turn.
// The sum over a tile's entries is a matrix product: with the weights
// separable, row (x, y) of A holds wx wy of entry k, column (component, z)
// of B holds wz F, and the 16 x 12 result is the tile's force.  Four entries
// are one 16x16x4 matrix instruction in the vertex real: per lane four LDS
// reads and two multiplies, where a lane per cell took 24 reads and 24
// fused multiply-adds for them (LDS reads bounded it).
// Bound by vector instructions where many tiles are touched (a tile of 25
// entries leaves lanes idle while their weights are formed), by latency on
// one cell.  400 800 vertices, FP32: 183 us with a lane per cell, 159 with
// the matrix instructions, 115 with one root per axis, the weights moved
// to their cells by conditional shifts and the keys ranked, not sorted.
// One launch (k_spread) holds two kinds of workgroups:
//   small: tiles with at most kSmallTile entries, kSparseTile where few
//          tiles are touched (off the touched-tile list, or all of them in
//          space order: spread_dense; the big ones are skipped), one wave
//          per tile, four independent waves
//          per workgroup, keys ranked against each other in LDS (up
//          to 64 entries are loaded as listed and staged in the column of
//          their rank, up to 128 put in order first), one running sum from
//          g in vertex order;
//   big:   the big-tile list, one workgroup of four waves per tile; each
//          wave sorts a run of 64 keys in registers and the runs are merged
//          by rank in LDS (a bitonic sort in LDS past 256 entries); wave w
//          sums the w-th contiguous quarter of the sorted list and the four
//          partial sums are added to g in wave order.
// Each clears the tile's count once done, so the next binning starts from
// zero without a clearing pass.
constexpr int kChunk = 32;
// LDS row of a staged chunk: the 16 (row, entry) words that a matrix operand
// reads at once, 4 rows of 4 entries, fall on 16 different banks
constexpr int kChunkRow = kChunk + 4;
constexpr int kSpreadWaves = 4;

// c += A B over four entries: lane l gives A[l % 16][l / 16] and
// B[l / 16][l % 16] and holds column l % 16 of c, four rows of it.  Rows are
// the tile's (x, y), 4 x + y; columns 4 component + z.
template <class R>
struct TileSum;
template <>
struct TileSum<float> {
    using V = float __attribute__((ext_vector_type(4)));
    __device__ static V add(float a, float b, V c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    __device__ static int x(int lane, int) { return lane >> 4; }
    __device__ static int y(int, int r) { return r; }
};
template <>
struct TileSum<double> {
    using V = double __attribute__((ext_vector_type(4)));
    __device__ static V add(double a, double b, V c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    __device__ static int x(int, int r) { return r; }
    __device__ static int y(int lane, int) { return lane >> 4; }
};

// Orders the LDS accesses of one wave (a wave's LDS operations complete in
// issue order; this keeps the compiler from moving them across).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Both kinds in one launch: workgroups [0, n_small) take the small tiles,
// the others the big ones.
template <class R>
struct SpreadArgs {
    LatView lv;
    Grid gd;
    int n_small;
    double h;
    // the touched-tile list (null: every tile is looked at, in space order)
    const int *active, *nactive, *big, *nbig;
    int ntiles, small;
    FastDiv dty, dtz;  // division by the tiles along y and z
    int* count;
    int cap;
    const int* list;
    const Vel4<R>* vp;  // the binning's position copies
    const R* vforce;
    NearView<R> nw;
    void* Fout;  // force field in the storage's force type
    int xcd;     // order of the small-tile workgroups over the XCDs (ibm_block)
};

// List entry `e` as loaded: the vertex's position copy and its force, two
// loads, where the stored base and weights were 60 B (FP32) on four lines.
// A near-wall vertex's kernel part carries the force times w (w < 1), its
// top-hat part the force times 1 - w (w > 0).
template <class R>
struct Entry {
    Vel4<R> P;
    R F[3];
    bool top;
};

template <class R>
__device__ __forceinline__ Entry<R> load_entry(const SpreadArgs<R>& A, int e)
{
    Entry<R> E;
    const bool nr = (e & kNearKey) != 0;
    const long v = nr ? (long)((e & ~kNearKey) >> 1) : (long)e;
    E.top = nr && (e & 1);
    E.P = A.vp[v];
    for (int k = 0; k < 3; ++k) E.F[k] = A.vforce[3 * v + k];
    if (nr) {
        const R wb = A.nw.blend[v];
        const bool scale = E.top ? wb > R(0) : wb < R(1);
        const R s = E.top ? R(1.) - wb : wb;
        if (scale)
            for (int k = 0; k < 3; ++k) E.F[k] *= s;
    }
    return E;
}

// Its weights on the tile's cells (rows 0-11: axis-major, 4 cells per axis)
// and its force (rows 12-14).
template <int SW, class R>
__device__ __forceinline__ void entry_weights(const SpreadArgs<R>& A, const int org[3], const Entry<R>& E, R ev[15])
{
    const Grid& gd = A.gd;
    const R x[3] = {E.P.x, E.P.y, E.P.z};
    const R h = A.nw.on && E.top ? R(1.0) : (R)A.h;
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        const int first = stencil_first(x[ax], h);
        const int b = stencil_base(first, gd.n[ax], gd.per[ax]);
        W4<R> w = axis_weights<SW, R>(x[ax], first);
        if (A.nw.on) {
            const W4<R> t = axis_weights<2, R>(x[ax], first);
            w = {E.top ? t.w0 : w.w0, E.top ? t.w1 : w.w1, E.top ? t.w2 : w.w2, E.top ? t.w3 : w.w3};
        }
        // the tile's first node past the stencil's; a stencil that wrapped
        // starts beyond the tile, and (but in a box of less than 8 nodes)
        // reaches it only past the face
        int d = org[ax] - b;
        if (gd.per[ax] && d < -3) d += gd.n[ax];
        R o[4];
        shifted<R>(w, d, o);
        if (gd.per[ax] && gd.n[ax] < 8) {  // both ends of a wrapped stencil may lie in one tile
            R u[4];
            shifted<R>(w, max(min(d + gd.n[ax], 4), -3), u);
#pragma unroll
            for (int l = 0; l < 4; ++l) o[l] = d + l < 0 ? (d + gd.n[ax] <= 3 ? u[l] : R(0)) : o[l];
        }
#pragma unroll
        for (int l = 0; l < 4; ++l) ev[4 * ax + l] = o[l];
    }
    for (int k = 0; k < 3; ++k) ev[12 + k] = E.F[k];
}

// Adds entries [0, cnt) of a staged half (cnt <= kChunk; the rows are zero
// from cnt to the half's end, so a padded entry adds nothing) in entry
// order, 16 at a time.
template <class R>
__device__ __forceinline__ void chunk_sum(const R (*ew)[kChunkRow], int cnt, int lane, typename TileSum<R>::V& acc)
{
    const int k = lane >> 4, i = (lane >> 2) & 3, j = lane & 3;
    const R *wx = ew[i] + k, *wy = ew[4 + j] + k, *wz = ew[8 + j] + k, *F = ew[12 + min(i, 2)] + k;
    for (int e = 0; e < cnt; e += 16) {
        R a[4], b[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            a[q] = wx[e + 4 * q] * wy[e + 4 * q];
            b[q] = wz[e + 4 * q] * F[e + 4 * q];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) acc = TileSum<R>::add(a[q], b[q], acc);
    }
}

// Adds the sorted entries [lo, hi) of a tile to acc, 64 at a time; key(e)
// gives the e-th sorted entry.
template <int SW, class R, class KeyOf>
__device__ __forceinline__ void sum_entries(const SpreadArgs<R>& A, const int org[3], int lo, int hi, KeyOf key,
                                            R (*ew)[kChunkRow], int lane, typename TileSum<R>::V& acc)
{
    for (int c0 = lo; c0 < hi; c0 += 64) {
        const int e = c0 + lane;
        R ev[15];
#pragma unroll
        for (int r = 0; r < 15; ++r) ev[r] = R(0.0);
        if (e < hi) entry_weights<SW, R>(A, org, load_entry<R>(A, key(e)), ev);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int cnt = min(kChunk, hi - c0 - half * kChunk);
            if (cnt <= 0) break;
            if ((lane >> 5) == half)
#pragma unroll
                for (int r = 0; r < 15; ++r) ew[r][lane & (kChunk - 1)] = ev[r];
            wave_sync();
            chunk_sum<R>(ew, cnt, lane, acc);
            wave_sync();
        }
    }
}

template <class R>
__device__ __forceinline__ void tile_origin(const SpreadArgs<R>& A, int t, int org[3])
{
    const unsigned rr = fdiv((unsigned)t, A.dtz), tx = fdiv(rr, A.dty);
    org[0] = (int)tx * kTile;
    org[1] = (int)(rr - tx * (unsigned)A.gd.nt[1]) * kTile;
    org[2] = (int)((unsigned)t - rr * (unsigned)A.gd.nt[2]) * kTile;
}

// The body force of a lane's column, the start of its sums.
template <class R>
__device__ __forceinline__ R column_start(const LatView& lv, int lane)
{
    const int i = (lane >> 2) & 3;
    return (R)(i == 0 ? lv.g[0] : (i == 1 ? lv.g[1] : lv.g[2]));
}

template <class FT, class R>
__device__ __forceinline__ void store_tile(const LatView& lv, const Grid& gd, const int org[3], int lane,
                                           typename TileSum<R>::V acc, FT* __restrict__ Fout)
{
    const int comp = (lane >> 2) & 3, z = org[2] + (lane & 3);
    if (comp == 3 || z >= gd.n[2]) return;
    FT* out = Fout + comp * lv.stride;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int x = org[0] + TileSum<R>::x(lane, r), y = org[1] + TileSum<R>::y(lane, r);
        if (x < gd.n[0] && y < gd.n[1]) out[(unsigned)((x * gd.n[1] + y) * gd.n[2] + z)] = (FT)acc[r];
    }
}

// How many of the n keys in LDS (padded to a multiple of 4 with keys that
// are below none) are below `mine`: four keys a read, the same address in
// every lane.
__device__ __forceinline__ int rank_in(const int* k, int n, int mine)
{
    int r = 0;
#pragma unroll 4
    for (int e = 0; e < n; e += 4) {
        const int4 q = *(const int4*)(k + e);
        r += (q.x < mine ? 1 : 0) + (q.y < mine ? 1 : 0) + (q.z < mine ? 1 : 0) + (q.w < mine ? 1 : 0);
    }
    return r;
}

// ascending bitonic sort of one key per lane across the wave
__device__ __forceinline__ int wave_sort(int key, int lane)
{
#pragma unroll
    for (int size = 2; size <= 64; size <<= 1)
#pragma unroll
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            const int other = __shfl_xor(key, stride);
            const bool up = (lane & size) == 0;
            const bool lower = (lane & stride) == 0;
            key = (lower == up) ? min(key, other) : max(key, other);
        }
    return key;
}

// number of entries of the ascending run r[0, 64) that are below `key`
__device__ __forceinline__ int rank_in_run(const int* r, int key)
{
    int lo = 0;  // count among r[0, 63), then r[63] when all of those are below
#pragma unroll
    for (int step = 32; step > 0; step >>= 1)
        if (r[lo + step - 1] < key) lo += step;
    return lo + (r[lo] < key ? 1 : 0);
}

template <class FT, int SW, class R>
__device__ __forceinline__ void spread_small(int blk, int nb, int* keys, R (*ew_all)[15][kChunkRow],
                                             const SpreadArgs<R>& A)
{
    const Grid& gd = A.gd;
    const int* __restrict__ active = A.active;
    int* __restrict__ count = A.count;
    const int* __restrict__ list = A.list;
    const int cap = A.cap;
    const int wv = threadIdx.x >> 6;
    R(*ew)[kChunkRow] = ew_all[wv];
    const int na = active ? *A.nactive : A.ntiles;
    const int lane = threadIdx.x & 63;
    const int stride = nb * kSpreadWaves;
    int a = blk * kSpreadWaves + wv;
    int t = a < na ? (active ? active[a] : a) : 0;
    while (a < na) {
        // the list's first slots are loaded with the count (not after it),
        // and the next tile's id while this one is summed
        const int raw = list[(long)t * cap + lane];
        const int n = count[t];
        const int a_next = a + stride;
        const int t_next = a_next < na ? (active ? active[a_next] : a_next) : 0;
        // a big tile is its workgroup's; a count already cleared (0) is one
        // that workgroup has finished (a listed tile has at least one entry)
        if (n > 64 && n <= A.small) {
            // two entries a lane: ordered through LDS, then 64 at a time
            const int raw1 = lane < n - 64 ? list[(long)t * cap + 64 + lane] : 0x7fffffff;
            int* k = keys + wv * kSmallTile;
            k[lane] = raw;
            k[64 + lane] = raw1;
            wave_sync();
            const int r0 = rank_in(k, n, raw), r1 = rank_in(k, n, raw1);
            wave_sync();
            k[r0] = raw;
            if (lane < n - 64) k[r1] = raw1;
            wave_sync();
            int org[3];
            tile_origin<R>(A, t, org);
            const R g = column_start<R>(A.lv, lane);
            typename TileSum<R>::V acc = {g, g, g, g};
            sum_entries<SW, R>(A, org, 0, n, [&](int e) { return k[e]; }, ew, lane, acc);
            store_tile<FT, R>(A.lv, gd, org, lane, acc, (FT*)A.Fout);
            if (lane == 0) count[t] = 0;
        } else if (n > 0 && n <= 64) {
            // lane e takes entry e as listed and stages it in the column of
            // its rank, so the loads do not wait for an order
            int org[3];
            tile_origin<R>(A, t, org);
            const R g = column_start<R>(A.lv, lane);
            typename TileSum<R>::V acc = {g, g, g, g};
            const bool live = lane < n;
            Entry<R> E = load_entry<R>(A, live ? raw : 0);
            int* k = keys + wv * kSmallTile;
            k[lane] = live ? raw : 0x7fffffff;
            wave_sync();
            const int rank = rank_in(k, n, raw);
            const int col = live ? rank : lane;
            if (!live) E.F[0] = E.F[1] = E.F[2] = R(0);
            R ev[15];
            entry_weights<SW, R>(A, org, E, ev);
            for (int h0 = 0; h0 < n; h0 += kChunk) {
                if ((col & ~(kChunk - 1)) == h0)
#pragma unroll
                    for (int r = 0; r < 15; ++r) ew[r][col & (kChunk - 1)] = ev[r];
                wave_sync();
                chunk_sum<R>(ew, min(kChunk, n - h0), lane, acc);
                wave_sync();
            }
            store_tile<FT, R>(A.lv, gd, org, lane, acc, (FT*)A.Fout);
            if (lane == 0) count[t] = 0;
        }
        a = a_next;
        t = t_next;
    }
}

template <class FT, int SW, class R>
__device__ __forceinline__ void spread_big(int blk, int nb, int* keys, int* runs, R (*ew_all)[15][kChunkRow],
                                           R (*part)[4][64], const SpreadArgs<R>& A)
{
    const Grid& gd = A.gd;
    int* __restrict__ count = A.count;
    const int* __restrict__ list = A.list;
    const int cap = A.cap;
    const int wv = threadIdx.x >> 6;
    R(*ew)[kChunkRow] = ew_all[wv];
    const int nt = *A.nbig;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    for (int a = blk; a < nt; a += nb) {
        const int t = A.big[a];
        const int n = min(count[t], cap);  // a longer list was cut at binning and reported there
        const long o = (long)t * cap;
        if (n <= 64 * kSpreadWaves) {
            // four register-sorted runs, merged by rank (keys are distinct)
            const int e = wv * 64 + lane;
            const int key = wave_sort(e < n ? list[o + e] : 0x7fffffff, lane);
            runs[e] = key;
            __syncthreads();
            if (e < n) {
                int r = lane;
#pragma unroll
                for (int w2 = 0; w2 < kSpreadWaves; ++w2)
                    if (w2 != wv) r += rank_in_run(runs + 64 * w2, key);
                keys[r] = key;
            }
        } else {
            int n2 = 1;
            while (n2 < n) n2 <<= 1;
            for (int k = tid; k < n2; k += blockDim.x) keys[k] = k < n ? list[o + k] : 0x7fffffff;
            __syncthreads();
            for (int size = 2; size <= n2; size <<= 1)
                for (int stride2 = size >> 1; stride2 > 0; stride2 >>= 1) {
                    for (int k = tid; k < n2; k += blockDim.x) {
                        const int partner = k ^ stride2;
                        if (partner > k) {
                            const bool up = (k & size) == 0;
                            const int a0 = keys[k], a1 = keys[partner];
                            if ((a0 > a1) == up) {
                                keys[k] = a1;
                                keys[partner] = a0;
                            }
                        }
                    }
                    __syncthreads();
                }
        }
        __syncthreads();
        int org[3];
        tile_origin<R>(A, t, org);
        // wave w sums the contiguous range [lo, hi) of the sorted entries
        const int q = (n + kSpreadWaves - 1) / kSpreadWaves;
        const int lo = min(n, wv * q), hi = min(n, lo + q);
        typename TileSum<R>::V acc = {R(0), R(0), R(0), R(0)};
        sum_entries<SW, R>(A, org, lo, hi, [&](int k) { return keys[k]; }, ew, lane, acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) part[wv][r][lane] = acc[r];
        __syncthreads();
        if (wv == 0) {
            const R g = column_start<R>(A.lv, lane);
            acc = {g, g, g, g};
#pragma unroll
            for (int w = 0; w < kSpreadWaves; ++w)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[r] += part[w][r][lane];
            store_tile<FT, R>(A.lv, gd, org, lane, acc, (FT*)A.Fout);
            if (lane == 0) count[t] = 0;
        }
        __syncthreads();  // keys and partial sums are rewritten for the next tile
    }
}

template <class S, int SW, class R>
__device__ __forceinline__ void spread_body(int bx, int nbx, const SpreadArgs<R>& A)
{
    using FT = typename Pop<S>::F;
    __shared__ __align__(16) int keys[kMaxList];
    __shared__ int runs[64 * kSpreadWaves];
    __shared__ R ew_all[kSpreadWaves][15][kChunkRow];
    __shared__ R part[kSpreadWaves][4][64];
    if (bx < A.n_small) spread_small<FT, SW, R>((int)ibm_block(bx, A.n_small, A.xcd), A.n_small, keys, ew_all, A);
    else spread_big<FT, SW, R>(bx - A.n_small, nbx - A.n_small, keys, runs, ew_all, part, A);
}

template <class S, int SW, class R>
__global__ void __launch_bounds__(64 * kSpreadWaves) k_spread(SpreadArgs<R> a)
{
    spread_body<S, SW, R>(blockIdx.x, gridDim.x, a);
}

// ------------------------------------------- stages paired in one launch
// Two stages of a coupled step that do not read each other's output run as
// one launch: workgroups [0, n1) take the first, the others the second
// (the choice is uniform over a workgroup, so its barriers stay whole).
// Binning | element forces: both read the positions only.
template <class R, BinForm FORM>
__global__ void __launch_bounds__(256) k_bin_elem(BinArgs<R> b, int n1, ElemArgs<R> e)
{
    const int bx = blockIdx.x;
    if (bx < n1) bin_group<R, FORM>(ibm_block(bx, n1, b.xcd), b);
    else elem_body<R>(ibm_block(bx - n1, (int)gridDim.x - n1, e.xcd), e);
}

// Vertex force gather (element forces) | velocity staging (the binning's
// tiles, the last collision's field).
template <class S, bool SWAPPED, bool EITHER, class R, int GL>
__global__ void __launch_bounds__(256) k_gather_stage(GatherArgs<R> ga, int n1, StageArgs sa)
{
    const int bx = blockIdx.x;
    if (bx < n1) gather_body<R, GL>(ibm_block(bx, n1, ga.xcd), ga);
    else stage_body<S, SWAPPED, EITHER>(bx - n1, gridDim.x - n1, sa);
}

// Spreading (lists, position copies and vertex forces) | interpolation +
// advection (position copies and staged velocity; it moves the vertices,
// which the spreading does not read).
template <class S, int SW, class R>
__global__ void __launch_bounds__(256) k_spread_interp(SpreadArgs<R> sp, int n1, InterpArgs<R> ia)
{
    const int bx = blockIdx.x;
    if (bx < n1) spread_body<S, SW, R>(bx, n1, sp);
    else interp_body<typename Pop<S>::C, SW, true, R>(bx - n1, (int)gridDim.x - n1, ia);
}

// ------------------------------------------------------- calibration
// shrink_rbc_volume (progs/common/calibrate_rbc_shape.h:13-72) with
// RBCParticle::relax_nodes (src/fsi/RBCParticle.hh:318-342) as its step,
// for every selected particle at once.  Node mass: area / 3 of each
// incident triangle (tri::triangle_area, src/fsi/TriangleUtils.h:52-55),
// summed in triangle order (the vertex's incidence list is in element
// order).  The step counter lives on the device so that the launches of
// any step are the same.
template <class R>
__global__ void __launch_bounds__(256) k_calib_mass(ForceView<R> f, long NV, const int* __restrict__ active,
                                                    double* __restrict__ mass, int* __restrict__ step)
{
#pragma clang fp contract(off)
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v == 0) *step += 1;
    if (v >= NV) return;
    const int p = f.v_part[v];
    if (!active[p]) return;
    const int s = f.p_shape[p];
    const long vo = f.p_voff[p];
    const long sv = f.s_voff[s] + (v - vo);
    const int* ht = f.s_vt_head + sv + s;
    const int* Lt = f.s_vt + f.s_vtoff[s] + ht[0];
    const int nt = ht[1] - ht[0];
    double M = 0.0;
    for (int k = 0; k < nt; ++k) {
        const long st = f.s_toff[s] + (Lt[k] >> 2);
        const D3 v0 = ld3d(f.pos + 3 * (vo + f.s_tri[3 * st])), v1 = ld3d(f.pos + 3 * (vo + f.s_tri[3 * st + 1])),
                 v2 = ld3d(f.pos + 3 * (vo + f.s_tri[3 * st + 2]));
        M += (0.5 * norm(cross(v1 - v0, v2 - v0))) / 3.;
    }
    mass[v] = M;
}

// One relax step of the selected particles: vel += F / M - damping vel,
// pos += vel; the first vertex of each sets vol_desired of this step (the
// ramp from vol_start to vol_final over the first n_it steps).  The step's
// arithmetic is FP64; the vertex state keeps the boundary's type.
template <class R>
__global__ void __launch_bounds__(256) k_calib_relax(long NV, const int* __restrict__ v_part,
                                                     const long* __restrict__ p_voff, const int* __restrict__ active,
                                                     const double* __restrict__ damping,
                                                     const double* __restrict__ vol_start,
                                                     const double* __restrict__ vol_final, int n_it,
                                                     const int* __restrict__ step, const double* __restrict__ mass,
                                                     const R* __restrict__ force, R* __restrict__ vel,
                                                     R* __restrict__ pos, double* __restrict__ params)
{
#pragma clang fp contract(off)
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= NV) return;
    const int p = v_part[v];
    if (!active[p]) return;
    const int it = *step - 1;
    if (v == p_voff[p] && it <= n_it)
        params[8 * p + 5] = vol_start[p] + ((double)it / (double)n_it) * (vol_final[p] - vol_start[p]);
    const double M = mass[v], d = damping[p];
    for (int k = 0; k < 3; ++k) {
        const double u0 = (double)vel[3 * v + k];
        const double u = u0 + ((double)force[3 * v + k] / M - d * u0);
        vel[3 * v + k] = (R)u;
        pos[3 * v + k] = (R)((double)pos[3 * v + k] + u);
    }
}

// --------------------------------------------------------------- motion
template <class R>
__global__ void k_move(long NV, R* __restrict__ pos, const R* __restrict__ vel)
{
    const long v = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= 3 * NV) return;
    pos[v] += vel[v];
}

// Per-particle area, signed volume and area-weighted centroid
// (src/fsi/DeformableParticle3D.hh:54-82) in FP64, by a fixed reduction
// order, so that the result does not depend on scheduling.  Every particle's
// triangles are cut into chunks of 256 (one workgroup each, a tree in LDS)
// and a second launch adds the chunk sums in chunk order; boundaries whose
// particles all have at most kGeomTriangles triangles take one launch of a
// workgroup per particle instead (k_geom: a lane's triangles one after the
// other, a butterfly per wave, the waves in order).  Both wait for memory:
// 1 280 triangles take 5.9 us in one launch, 4.5 + 4.6 in two, but 5 120
// take 13 (with 512 or 1 024 lanes alike) against 9.2, and 18 cells of them
// 17 against 9.9.
constexpr long kGeomTriangles = 2048;
template <class R>
struct GeomArgs {
    ForceView<R> f;
    const int2* chunks;
    const int* t_vert;
    double* partial;
    int nchunk, np;
    Grid gd;
    const int* p_choff;
    const long* p_voff;
    double *geom, *delta;
    R* pos;
    int remap;
    const int* p_model;
};

// Adds one triangle's share to the sums: its area, six times its volume and
// three times its area-weighted centroid (the quotients are taken once per
// particle, in geom_store: four FP64 divisions were half of a triangle's
// instructions).
template <class R>
__device__ __forceinline__ void triangle_sums(const R* pos, const int* tv, double acc[kGeomSums])
{
    const D3 v0 = ld3d(pos + 3 * (long)tv[0]), v1 = ld3d(pos + 3 * (long)tv[1]), v2 = ld3d(pos + 3 * (long)tv[2]);
    const double dA = 0.5 * norm(cross(v1 - v0, v2 - v0));
    acc[0] += dA;
    acc[1] += dot(v0, cross(v1, v2));
    acc[2] += (v0.x + v1.x + v2.x) * dA;
    acc[3] += (v0.y + v1.y + v2.y) * dA;
    acc[4] += (v0.z + v1.z + v2.z) * dA;
}

// Chunk c (its row of `chunks`: first triangle, triangles, global indices)
// -> its sums.
template <class R>
__device__ __forceinline__ void geom_partial_body(int c, const GeomArgs<R>& A)
{
    const ForceView<R>& f = A.f;
    const int2* __restrict__ chunks = A.chunks;
    const int* __restrict__ t_vert = A.t_vert;
    double* __restrict__ partial = A.partial;
    __shared__ double sh[kGeomSums][256];
    const int2 ch = chunks[c];
    double acc[kGeomSums] = {0, 0, 0, 0, 0};
    if ((int)threadIdx.x < ch.y) triangle_sums<R>(f.pos, t_vert + 3 * ((long)ch.x + threadIdx.x), acc);
    for (int q = 0; q < kGeomSums; ++q) sh[q][threadIdx.x] = acc[q];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int q = 0; q < kGeomSums; ++q) sh[q][threadIdx.x] += sh[q][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x < kGeomSums) partial[kGeomSums * (long)c + threadIdx.x] = sh[threadIdx.x][0];
}

template <class R>
__global__ void __launch_bounds__(256) k_geom_partial(GeomArgs<R> a) { geom_partial_body<R>(blockIdx.x, a); }

// A particle's sums -> geometry (one lane); the centre of mass is then
// mapped onto the periodic grid (src/fsi/ParticleBase.hh:113-136,
// src/fsi/Periodicity.h:83-87), `sft` the shift of the whole particle.
template <class R>
__device__ __forceinline__ void geom_store(int p, const GeomArgs<R>& A, const double acc[kGeomSums], double sft[3])
{
    const Grid& gd = A.gd;
    double* G = A.geom + kGeomSums * p;
    const double area = acc[0];
    const double a3 = 3.0 * area;
    const double com[3] = {acc[2] / a3, acc[3] / a3, acc[4] / a3};
    G[0] = area;
    G[1] = acc[1] / 6.;
    for (int d = 0; d < 3; ++d) {
        sft[d] = 0.0;
        G[2 + d] = com[d];
        // a rigid particle maps its own centre of mass (rigid.hip)
        if (A.remap && gd.per[d] && A.p_model[p] != BL_MODEL_RIGID) {
            const double L = (double)gd.n[d];
            const double x0 = -0.5;
            const double r = com[d] - L * floor((com[d] - x0) * (1. / L));
            sft[d] = r - com[d];
            G[2 + d] = r;
        }
        A.delta[3 * p + d] = sft[d];
    }
}

// The shift of a whole particle by its workgroup.
template <class R>
__device__ __forceinline__ void geom_shift(int p, const GeomArgs<R>& A, const double sft[3])
{
    const double s0 = sft[0], s1 = sft[1], s2 = sft[2];
    if (s0 == 0.0 && s1 == 0.0 && s2 == 0.0) return;
    for (long v = A.p_voff[p] + threadIdx.x; v < A.p_voff[p + 1]; v += blockDim.x) {
        A.pos[3 * v] = (R)((double)A.pos[3 * v] + s0);
        A.pos[3 * v + 1] = (R)((double)A.pos[3 * v + 1] + s1);
        A.pos[3 * v + 2] = (R)((double)A.pos[3 * v + 2] + s2);
    }
}

// Chunk partials -> geometry.
template <class R>
__device__ __forceinline__ void geom_final_body(int p, const GeomArgs<R>& A)
{
    const int* __restrict__ p_choff = A.p_choff;
    const double* __restrict__ partial = A.partial;
    __shared__ double sft[3];
    __shared__ double part[64][kGeomSums];  // a batch of chunk partials, loaded by all lanes at once
    const int c0 = p_choff[p], c1 = p_choff[p + 1];
    double acc[kGeomSums] = {0, 0, 0, 0, 0};
    for (int b = c0; b < c1; b += 64) {
        const int nb = min(64, c1 - b);
        if ((int)threadIdx.x < nb)
            for (int q = 0; q < kGeomSums; ++q)
                part[threadIdx.x][q] = partial[kGeomSums * (long)(b + threadIdx.x) + q];
        __syncthreads();
        if (threadIdx.x == 0)
            for (int k = 0; k < nb; ++k)  // chunk order
                for (int q = 0; q < kGeomSums; ++q) acc[q] += part[k][q];
        __syncthreads();
    }
    if (threadIdx.x == 0) geom_store(p, A, acc, sft);
    __syncthreads();
    geom_shift(p, A, sft);
}

// One particle by one workgroup of kGeomBlock lanes: lane t takes triangles
// t, t + kGeomBlock, ... in order, then a butterfly per wave and the waves
// in order.
constexpr int kGeomBlock = 512;

template <class R>
__device__ __forceinline__ void geom_body(int p, const GeomArgs<R>& A)
{
    __shared__ double wave[kGeomBlock / 64][kGeomSums];
    __shared__ double sft[3];
    const int tid = threadIdx.x;
    double acc[kGeomSums] = {0, 0, 0, 0, 0};
#pragma unroll 4
    for (long t = A.f.p_toff[p] + tid; t < A.f.p_toff[p + 1]; t += kGeomBlock)
        triangle_sums<R>(A.f.pos, A.t_vert + 3 * t, acc);
    for (int o = 1; o < 64; o <<= 1)
#pragma unroll
        for (int q = 0; q < kGeomSums; ++q) acc[q] += __shfl_xor(acc[q], o);
    if ((tid & 63) == 0)
        for (int q = 0; q < kGeomSums; ++q) wave[tid >> 6][q] = acc[q];
    __syncthreads();
    if (tid == 0) {
        for (int k = 1; k < kGeomBlock / 64; ++k)
            for (int q = 0; q < kGeomSums; ++q) acc[q] += wave[k][q];
        geom_store(p, A, acc, sft);
    }
    __syncthreads();
    geom_shift(p, A, sft);
}

template <class R>
__global__ void __launch_bounds__(kGeomBlock) k_geom(GeomArgs<R> a) { geom_body<R>(blockIdx.x, a); }

template <class R>
__global__ void __launch_bounds__(64) k_geom_final(GeomArgs<R> a) { geom_final_body<R>(blockIdx.x, a); }

// --------------------------------------------------------- voxelization
// z-rays through integer (x, y) columns (RayTracer::find_intersections_z,
// src/fsi/RayTracer.hh:19-39,80-108; z mapped into [-0.5, nz - 0.5) on a
// periodic z axis, as ZBuffer::put does, src/fsi/ZBuffer.h:39-49), then the
// fill of apply_voxelization (src/fsi/ImmersedBoundaryDynamics_voxelization.hh:
// 121-165): between consecutive sorted hits the nodes alternate outside and
// inside, a later segment overwriting a shared end node.  A node is
// therefore inside when an odd number of hits lie at or below it, and the
// hits of a column need neither a list nor an order: each toggles the bit of
// the first node at or above it, and the fill takes the parity of the bits
// up to a node.  Only the last node differs: the fill's tail runs where the
// last hit's first node comes before it, so with that hit between the last
// two nodes the last one keeps its value, and with a hit exactly on it it
// takes the value before that hit; a flag word per column says so.
// Bound by latency.  As hit counts, a scan, a second trace into lists and a
// sort per column this was six launches and 44 us for 5 120 triangles on 75
// x 61 columns of 83 nodes; two launches and 9.4 us.
constexpr int kFillCols = 16;  // columns a workgroup fills
constexpr unsigned kHitBeyond = 1, kHitOnLast = 2, kHitBeforeLast = 4;

__host__ __device__ inline int column_words(int nz) { return (nz + 31) / 32 + 1; }

// One triangle's hits into the columns' bits; returns their number.
template <class R>
__device__ __forceinline__ int trace_triangle(const ForceView<R>& f, const Grid& gd, long g, long NT, unsigned* bits)
{
    if (g >= NT) return 0;
    const int p = f.t_part[g];
    const int s = f.p_shape[p];
    const long vo = f.p_voff[p];
    const int* tri = f.s_tri + 3 * (f.s_toff[s] + (g - f.p_toff[p]));
    const D3 a = ld3d(f.pos + 3 * (vo + tri[0])), b = ld3d(f.pos + 3 * (vo + tri[1])),
             c = ld3d(f.pos + 3 * (vo + tri[2]));
    // a triangle with a non-finite corner, or wider than the lattice, is
    // not traced (its membrane diverged; the binning reports it)
    const double ext = fmax(fmax(fabs(a.x), fabs(b.x)), fmax(fmax(fabs(c.x), fabs(a.y)), fmax(fabs(b.y), fabs(c.y))));
    if (!(ext < 1e9)) return 0;
    const long x0 = (long)ceil(fmin(a.x, fmin(b.x, c.x))), x1 = (long)floor(fmax(a.x, fmax(b.x, c.x)));
    const long y0 = (long)ceil(fmin(a.y, fmin(b.y, c.y))), y1 = (long)floor(fmax(a.y, fmax(b.y, c.y)));
    if (x1 - x0 > (long)gd.n[0] + 4 || y1 - y0 > (long)gd.n[1] + 4) return 0;
    const D3 e1 = b - a, e2 = c - a;
    const D3 dir = {0, 0, 1};
    const D3 q = cross(dir, e2);
    const double det = dot(e1, q);
    if (fabs(det) < 2.220446049250313e-16) return 0;
    const double fi = 1 / det;
    const int W = column_words(gd.n[2]);
    int hits = 0;
    for (long i = x0; i <= x1; ++i)
        for (long j = y0; j <= y1; ++j) {
            const D3 o = {(double)i, (double)j, 0.};
            const D3 sv = o - a;
            const double u = fi * dot(sv, q);
            if (u < 0.0) continue;
            const D3 r = cross(sv, e1);
            const double v = fi * dot(dir, r);
            if (v < 0.0 || u + v > 1.0) continue;
            const int cx_ = wrap_node((int)i, gd.n[0], gd.per[0]);
            const int cy_ = wrap_node((int)j, gd.n[1], gd.per[1]);
            if (cx_ < 0 || cy_ < 0) continue;
            const long col = (long)cx_ * gd.n[1] + cy_;
            double z = fi * dot(e2, r);
            if (gd.per[2]) {
                const double L = (double)gd.n[2];
                z = z - L * floor((z + 0.5) * (1. / L));
            }
            ++hits;
            const int last = gd.n[2] - 1;
            unsigned* b = bits + col * W;
            if (z > (double)last) {
                atomicOr(&b[W - 1], kHitBeyond);
                continue;
            }
            const double node = fmax(ceil(z), 0.0);
            const int k = (int)node;
            atomicXor(&b[k >> 5], 1u << (k & 31));
            if (ceil(z) == (double)last) atomicOr(&b[W - 1], z == (double)last ? kHitOnLast : kHitBeforeLast);
        }
    return hits;
}

template <class R>
__global__ void __launch_bounds__(256) k_ray_hits(ForceView<R> f, Grid gd, long NT, unsigned* bits, int* total)
{
    __shared__ int hits;
    if (threadIdx.x == 0) hits = 0;
    __syncthreads();
    const int n = trace_triangle<R>(f, gd, (long)blockIdx.x * blockDim.x + threadIdx.x, NT, bits);
    if (n) atomicAdd(&hits, n);
    __syncthreads();
    if (threadIdx.x == 0 && hits) atomicAdd(total, hits);
}
// Fills kFillCols columns per workgroup, a lane per node (consecutive bytes),
// and clears their bits for the next step.  `cap`: the most hits a step may
// have; more than 64 per triangle are those of a membrane torn far beyond
// its lattice, and are reported.
__global__ void __launch_bounds__(256) k_fill_columns(Grid gd, unsigned* bits, int* total, long cap, int* status,
                                                      unsigned char* phase)
{
    const int nz = gd.n[2], W = column_words(nz);
    const long ncol = (long)gd.n[0] * gd.n[1], c0 = (long)blockIdx.x * kFillCols;
    const int nc = (int)(ncol - c0 < kFillCols ? ncol - c0 : kFillCols);
    unsigned* b = bits + c0 * W;
    for (int i = threadIdx.x; i < nc * nz; i += blockDim.x) {
        const int col = (int)((unsigned)i / (unsigned)nz), z = i - col * nz;
        const unsigned* w = b + col * W;
        unsigned x = w[z >> 5] & (0xffffffffu >> (31 - (z & 31)));
        for (int k = 0; k < (z >> 5); ++k) x ^= w[k];
        unsigned char in = __popc(x) & 1;
        if (z == nz - 1) {
            const unsigned fl = w[W - 1];
            if (!(fl & kHitBeyond)) {
                if (fl & kHitOnLast) in ^= 1;
                else if (fl & kHitBeforeLast) continue;
            }
        }
        phase[c0 * nz + i] = in;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nc * W; i += blockDim.x) b[i] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (*total > cap) atomicOr(&status[2], 2);
        *total = 0;
    }
}

}  // namespace

// ======================================================== host helpers
namespace {

template <class T>
int upload(T*& dst, const std::vector<T>& src)
{
    hipFree(dst);
    dst = nullptr;
    const size_t n = std::max<size_t>(src.size(), 1);
    BL_HIP(hipMalloc(&dst, n * sizeof(T)));
    if (!src.empty()) BL_HIP(hipMemcpy(dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice));
    return BL_OK;
}

template <class T>
int alloc(T*& dst, size_t n)
{
    hipFree(dst);
    dst = nullptr;
    BL_HIP(hipMalloc(&dst, std::max<size_t>(n, 1) * sizeof(T)));
    return BL_OK;
}

int alloc_bytes(void*& dst, size_t n)
{
    hipFree(dst);
    dst = nullptr;
    BL_HIP(hipMalloc(&dst, std::max<size_t>(n, 1)));
    return BL_OK;
}

// Runs fn(R{}) with R the boundary's vertex real type.
template <class Fn>
auto with_vreal(bl_ibm g, Fn&& fn)
{
    if (g->vreal == 4) return fn(float{});
    return fn(double{});
}

// The vertex real type that goes with a population storage type.
template <class S>
struct VRof {
    using T = float;
};
template <>
struct VRof<double> {
    using T = double;
};

// The kernels templated on the storage use its vertex type; a boundary
// whose vertex type differs (rigid particles on a reduced-precision
// lattice) never reaches them (rigid_refuse_coupling).
int vreal_matches_storage(bl_ibm g)
{
    const int want = g->lat->storage == BL_STORE_F64 ? 8 : 4;
    if (g->vreal != want)
        return fail(BL_ERR_STATE, "immersed boundary: vertex precision does not match the lattice storage");
    return BL_OK;
}

template <class R>
ForceView<R> force_view(bl_ibm g)
{
    ForceView<R> f;
    f.np = g->np;
    f.p_voff = g->p_voff; f.p_toff = g->p_toff; f.p_loff = g->p_loff; f.p_poff = g->p_poff;
    f.p_shape = g->p_shape; f.p_model = g->p_model; f.p_bug = g->p_bug;
    f.p_params = g->p_params; f.p_geom = g->p_geom;
    f.s_voff = g->s_voff; f.s_toff = g->s_toff; f.s_loff = g->s_loff; f.s_poff = g->s_poff;
    f.s_vtoff = g->s_vtoff; f.s_vloff = g->s_vloff; f.s_vpoff = g->s_vpoff;
    f.s_tri = g->s_tri; f.s_tri_area0 = g->s_tri_area0; f.s_tri_geo0 = g->s_tri_geo0;
    f.s_link = g->s_link; f.s_link_len = g->s_link_len;
    f.s_pair = g->s_pair; f.s_pair_cs0 = g->s_pair_cs0;
    f.s_vt_head = g->s_vt_head; f.s_vt = g->s_vt;
    f.s_vl_head = g->s_vl_head; f.s_vl = g->s_vl;
    f.s_vp_head = g->s_vp_head; f.s_vp = g->s_vp;
    f.s_area0 = g->s_area0;
    f.pos = (const R*)g->pos;
    f.v_part = g->v_part; f.t_part = g->t_part; f.r_part = g->r_part; f.l_part = g->l_part;
    f.v_inc = (const int4*)g->v_inc;
    return f;
}

template <class R>
NearView<R> near_view(bl_ibm g)
{
    NearView<R> nw;
    nw.b = g->boundary;
    nw.on = g->has_boundary && g->v_near ? 1 : 0;
    nw.near = g->v_near;
    nw.blend = (R*)g->v_blend;
    return nw;
}

// Per-vertex near-wall buffers, once both a boundary and the vertices exist.
int alloc_near(bl_ibm g)
{
    if (!g->has_boundary || !g->inited || g->v_near) return BL_OK;
    const size_t nv = (size_t)std::max<long>(g->NV, 1);
    hipError_t e = hipMalloc(&g->v_near, nv);
    if (e == hipSuccess) e = hipMalloc(&g->v_blend, (size_t)g->vreal * nv);
    if (e != hipSuccess) return fail(BL_ERR_HIP, std::string("near-wall buffers: ") + hipGetErrorString(e));
    return BL_OK;
}

inline unsigned nblk(long n, int b = 256) { return (unsigned)((n + b - 1) / b); }

int need_init(bl_ibm g)
{
    if (!g) return fail(BL_ERR_ARG, "null ibm handle");
    if (!g->inited) return fail(BL_ERR_STATE, "immersed boundary not initialised (call bl_ibm_init)");
    if (!g->lat) return fail(BL_ERR_STATE, "the lattice of this immersed boundary was destroyed");
    return BL_OK;
}

void mark(bl_ibm g, int k)
{
    if (g->timing) hipEventRecord(g->ev[k], g->lat->stream);
}

template <class R>
GeomArgs<R> geom_args(bl_ibm g, int remap)
{
    GeomArgs<R> a;
    a.f = force_view<R>(g);
    a.chunks = (const int2*)g->ch_tab;
    a.t_vert = g->t_vert;
    a.partial = g->ch_partial;
    a.nchunk = g->nchunk;
    a.np = g->np;
    a.gd = grid_of(g->lat);
    a.p_choff = g->p_choff;
    a.p_voff = g->p_voff;
    a.geom = g->p_geom;
    a.delta = g->p_delta;
    a.pos = (R*)g->pos;
    a.remap = remap;
    a.p_model = g->p_model;
    return a;
}

int update_particles(bl_ibm g, int remap, hipStream_t s)
{
    if (g->np == 0) return BL_OK;
    with_vreal(g, [&](auto tag) {
        using R = decltype(tag);
        const GeomArgs<R> a = geom_args<R>(g, remap);
        if (g->geom_one) {
            hipLaunchKernelGGL(k_geom<R>, dim3(g->np), dim3(kGeomBlock), 0, s, a);
            return 0;
        }
        hipLaunchKernelGGL(k_geom_partial<R>, dim3(g->nchunk), dim3(256), 0, s, a);
        hipLaunchKernelGGL(k_geom_final<R>, dim3(g->np), dim3(64), 0, s, a);
        return 0;
    });
    BL_CHECK_LAUNCH();
    return BL_OK;
}

int update_particles(bl_ibm g, int remap) { return update_particles(g, remap, g->lat->stream); }

// Stencil binning into the tile lists, the touched-tile list and the force
// flags of this step (buffer g->alt), on stream s.  The spreading kernels
// clear the counts of the tiles they consume; a binning that no spreading
// consumed leaves them set, and the next one clears first.  `done`
// (optional) is recorded once the lists are complete.
//
// Before it, list g->alt and flag buffer flags_alt are readied: counters a
// binning left unconsumed are cleared, the flags of the tiles the list held
// (two steps back) are cleared and the list emptied.  That may run as soon
// as the last staging has read those flags, carried by the interpolation
// launch of the step before (prep_rare + list_reset_of), or here.
ListReset list_reset_of(bl_ibm g)
{
    bl_lattice L = g->lat;
    ListReset lr;
    lr.act = g->active + (long)g->alt * L->ntiles;
    lr.na = g->n_active + g->alt;
    lr.flags = g->flags_alt;
    lr.pairs = g->n_active + 5 + g->alt;
    lr.arrive = g->n_active + 4;
    lr.nbig = g->n_active + 8 + g->alt;
    return lr;
}

void prep_rare(bl_ibm g, hipStream_t s)
{
    bl_lattice L = g->lat;
    if (g->bins_dirty) {
        hipLaunchKernelGGL(k_clear_bins, dim3(nblk(L->ntiles)), dim3(256), 0, s, g->tile_count, L->ntiles);
        g->bins_dirty = false;
    }
    if (g->alt_full) {
        hipLaunchKernelGGL(k_zero_u8, dim3(nblk(L->ntiles)), dim3(256), 0, s, g->flags_alt, L->ntiles);
        g->alt_full = false;
    }
}

int prep_bin(bl_ibm g, hipStream_t s)
{
    prep_rare(g, s);
    hipLaunchKernelGGL(k_bin_prep, dim3((unsigned)std::min<long>(nblk(g->lat->ntiles), kResetBlocks)), dim3(256), 0, s,
                       list_reset_of(g));
    BL_CHECK_LAUNCH();
    g->prepped = true;
    return BL_OK;
}

// With more vertices than tiles, about half the tiles or more are touched.
// The spreading's waves then walk all of them in space order, sixteen
// workgroups after one another on an XCD (the touched-tile list's order is
// the binning's arrival), and a wave takes tiles of up to 128 entries: of
// the 171 x 70 x 101 suspension's, spreading | interpolation 50.2 -> 46.6
// us, and fewer tiles queue on the big-tile list's counter (binning of the
// 400-cell one 100 -> 88 us).  One cell touches a few hundred tiles, fewer
// than there are CUs for: there four waves take a tile past 64 entries
// (2 562 vertices: 11.6 us against 15.7).
bool spread_dense(bl_ibm g) { return g->NV >= g->lat->ntiles; }

// Below this many vertices a stage is a few workgroups, and its time is the
// launch: stages that do not read each other's output then share one.
constexpr long kPairedVertices = 65536;
bool use_pairs(bl_ibm g) { return g->NV > 0 && g->NV < kPairedVertices; }

template <class R>
BinArgs<R> bin_args(bl_ibm g)
{
    bl_lattice L = g->lat;
    BinArgs<R> a;
    a.gd = grid_of(L);
    a.S = g->S;
    a.h = g->h;
    a.NV = g->NV;
    a.pos = (const R*)g->pos;
    a.vp = (Vel4<R>*)g->v_pos0;
    a.count = g->tile_count;
    a.list = g->tile_list;
    a.cap = kTileCap;
    a.act = g->active + (long)g->alt * L->ntiles;
    a.na = g->n_active + g->alt;
    a.flags = g->flags_alt;
    a.status = g->n_active;
    a.pairs = g->n_active + 5 + g->alt;
    a.big = g->active + (2L + g->alt) * L->ntiles;
    a.nbig = g->n_active + 8 + g->alt;
    a.small = spread_dense(g) ? kSmallTile : kSparseTile;
    a.nw = near_view<R>(g);
    a.xcd = g->lp[BL_IBM_XCD];
    return a;
}

// workgroups of a binning with bb threads each
int bin_blocks(bl_ibm g, int bb, bool many) { return (int)nblk(g->NV, bb / kBinLanes * (many ? kBinMany : 1)); }

bool bin_many(bl_ibm g)
{
    return g->NV >= kManyAny || (g->NV >= kManyVertices && g->NV <= kMeshVertices * g->np);
}

// f(form, workgroups) with the boundary's form of binning
template <class F>
void with_bin_form(bl_ibm g, int bb, F f)
{
    const bool many = bin_many(g);
    const int nb = bin_blocks(g, bb, many);
    if (many && g->has_boundary && g->v_near) f(std::integral_constant<BinForm, BIN_MANY_NEAR>{}, nb);
    else if (many) f(std::integral_constant<BinForm, BIN_MANY>{}, nb);
    else f(std::integral_constant<BinForm, BIN_ONE>{}, nb);
}

// host state after a binning has been enqueued
void binned(bl_ibm g)
{
    g->binned = true;
    g->bins_dirty = true;
    g->last_list = g->alt;
}

int do_bin(bl_ibm g, hipStream_t s, hipEvent_t done = nullptr)
{
    int rc;
    if (!g->prepped && (rc = prep_bin(g, s))) return rc;
    g->prepped = false;
    if (g->NV)
        with_vreal(g, [&](auto tag) {
            using R = decltype(tag);
            const int bb = g->lp[BL_IBM_BIN_BLOCK];
            with_bin_form(g, bb, [&](auto form, int nb) {
                hipLaunchKernelGGL((k_bin<R, decltype(form)::value>), dim3(nb), dim3(bb), 0, s, bin_args<R>(g));
            });
            return 0;
        });
    if (done) BL_HIP(hipEventRecord(done, s));
    BL_CHECK_LAUNCH();
    binned(g);
    return BL_OK;
}

LatView ibm_view(bl_ibm g)
{
    LatView lv = view_of(g->lat);
    if (!g->lat->force_field) lv.flags = nullptr;
    return lv;
}

// Where the staging takes the touched tiles off their list: few of many.
// By cells, every cell looks at its tile's flag (1.6 us for 10^6 cells) and
// the touched ones load whole lines; off the list a wave loads a tile's 4 x
// 4 rows of 4, a part of each line, 1.5 to 4.5 ns a tile more.  Steps with
// NV vertices per tile, by cells | off the list: 384^3 FP64 0.01, the pass
// alone 86 | 24 us; 300 x 200 x 190 0.11 FP64 784 | 775, FP16s 260 | 248;
// 256 x 256 x 128 0.16 FP32 304 | 295, 0.49 389 | 403; 256 x 128 x 128 0.08
// FP64 273 | 261, FP16s 90 | 87, 0.31 FP32 181 | 183, FP16s 114 | 123; on
// fewer cells nothing to gain (128^3 FP32 0.02 74 | 74, 0.63 106 | 121).
bool stage_by_list(bl_ibm g)
{
    const long n = g->lat->ncell;
    return n >= 1l << 22 && g->NV * (n >= 1l << 23 ? 4 : 8) <= g->lat->ntiles;
}

// Velocity staging of the step whose binning is the last one, before that
// binning's spreading: the last collision's force field and flags are the
// lattice's, and the binning's flags are in flags_alt.
StageArgs stage_args(bl_ibm g)
{
    bl_lattice L = g->lat;
    StageArgs a;
    a.lv = ibm_view(g);
    a.touched = g->flags_alt;
    a.ut = g->ut;
    a.active = stage_by_list(g) ? g->active + (long)g->last_list * L->ntiles : nullptr;
    a.nactive = g->n_active + g->last_list;
    a.dty = make_fastdiv((unsigned)L->nty);
    a.dtz = make_fastdiv((unsigned)L->ntz);
    return a;
}

// u on the cells of the touched tiles: a thread per cell, or about a wave
// per touched tile (at most every tile, and fewer than the vertices for a
// membrane; a wave that finds more takes several)
unsigned stage_blocks(bl_ibm g, bool list)
{
    if (!list) return (unsigned)((g->lat->ncell + 255) / 256);
    return (unsigned)std::max<long>(1, std::min<long>(std::min<long>(g->lat->ntiles, g->NV) / 4 + 1, 2048));
}

template <class S>
void launch_stage_s(const StageArgs& a, unsigned nblocks, bool swapped, hipStream_t s)
{
    if (swapped)
        hipLaunchKernelGGL((k_stage_u<S, true>), dim3(nblocks), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((k_stage_u<S, false>), dim3(nblocks), dim3(256), 0, s, a);
}

int launch_stage(bl_ibm g, hipStream_t s)
{
    bl_lattice L = g->lat;
    if (g->NV == 0) return BL_OK;
    const StageArgs a = stage_args(g);
    const bool swapped = (L->steps & 1) != 0;
    const unsigned nb = stage_blocks(g, a.active != nullptr);
    if (L->storage == BL_STORE_F64) launch_stage_s<double>(a, nb, swapped, s);
    else if (L->storage == BL_STORE_F32) launch_stage_s<float>(a, nb, swapped, s);
    else launch_stage_s<__half>(a, nb, swapped, s);
    BL_CHECK_LAUNCH();
    return BL_OK;
}

template <class R>
InterpArgs<R> interp_args(bl_ibm g, const ListReset& lr)
{
    InterpArgs<R> a;
    a.gd = grid_of(g->lat);
    a.h = g->h;
    a.NV = g->NV;
    a.vp = (const Vel4<R>*)g->v_pos0;
    a.ut = g->ut;
    a.vel = (R*)g->vel;
    a.pos = (R*)g->pos;
    a.lr = lr;
    a.nw = near_view<R>(g);
    a.xcd = g->lp[BL_IBM_XCD];
    return a;
}

unsigned interp_blocks(bl_ibm g, int blk = 256) { return (unsigned)nblk((g->S == 2 ? 4 : 16) * g->NV, blk); }

template <class C, bool MOVE>
void launch_interp_c(bl_ibm g, hipStream_t s, const ListReset& lr)
{
    using R = C;  // the staged velocity's type is the vertex type
    const InterpArgs<R> a = interp_args<R>(g, lr);
    const int ib = g->lp[BL_IBM_INTERP_BLOCK];
    const dim3 grid(interp_blocks(g, ib));
    if (g->S == 4) hipLaunchKernelGGL((k_interp<C, 4, MOVE, R>), grid, dim3(ib), 0, s, a);
    else if (g->S == 3) hipLaunchKernelGGL((k_interp<C, 3, MOVE, R>), grid, dim3(ib), 0, s, a);
    else hipLaunchKernelGGL((k_interp<C, 2, MOVE, R>), grid, dim3(ib), 0, s, a);
}

// The list reset carried by a launch that follows this step's spreading:
// the flags and list of two steps back are free once the staging has read
// them.
ListReset reset_next_of(bl_ibm g, hipStream_t s)
{
    prep_rare(g, s);
    g->prepped = true;
    return list_reset_of(g);
}

// vertex velocities from the staged u; with `move` the vertices advance.
// `reset_next` (after this step's spreading, once its staging is done):
// the launch also readies the list of the next binning.
int launch_interp(bl_ibm g, bool move, hipStream_t s, bool reset_next = false)
{
    if (g->NV == 0) return BL_OK;
    int rc = vreal_matches_storage(g);
    if (rc) return rc;
    ListReset lr;
    if (reset_next) lr = reset_next_of(g, s);
    const bool f64 = g->lat->storage == BL_STORE_F64;
    if (f64 && move) launch_interp_c<double, true>(g, s, lr);
    else if (f64) launch_interp_c<double, false>(g, s, lr);
    else if (move) launch_interp_c<float, true>(g, s, lr);
    else launch_interp_c<float, false>(g, s, lr);
    BL_CHECK_LAUNCH();
    return BL_OK;
}

// Spreading of the last binning's lists into the boundary's second force
// buffer; `blocks` receives the launch's workgroup count.
// `share`: boxes whose spreading shares one launch (a batched ensemble);
// the grid's lower bounds are divided among them.
template <class R>
SpreadArgs<R> spread_args(bl_ibm g, unsigned& blocks, int share = 1)
{
    bl_lattice L = g->lat;
    SpreadArgs<R> a;
    a.lv = ibm_view(g);
    a.gd = grid_of(L);
    a.h = g->h;
    const bool dense = spread_dense(g);
    a.small = dense ? kSmallTile : kSparseTile;
    a.dty = make_fastdiv((unsigned)L->nty);
    a.dtz = make_fastdiv((unsigned)L->ntz);
    a.active = dense ? nullptr : g->active + (long)g->alt * L->ntiles;
    a.ntiles = (int)L->ntiles;
    a.nactive = g->n_active + g->alt;
    a.big = g->active + (2L + g->alt) * L->ntiles;
    a.nbig = g->n_active + 8 + g->alt;
    a.count = g->tile_count;
    a.cap = kTileCap;
    a.list = g->tile_list;
    a.vp = (const Vel4<R>*)g->v_pos0;
    a.vforce = (const R*)g->force;
    a.nw = near_view<R>(g);
    a.Fout = g->force_alt;
    a.xcd = g->lp[BL_IBM_XCD] == 0 && dense ? 4 : g->lp[BL_IBM_XCD];
    // about one small-tile wave per touched tile and one workgroup per big
    // tile: the touched tiles are at most every tile and, for membranes,
    // fewer than the vertices (by default a wave per vertex); big tiles
    // fewer than a 32nd of the vertices (by default a workgroup per 32
    // vertices).  Both are launch parameters: the grid does not change any
    // sum.
    const long sw = (long)g->NV * g->lp[BL_IBM_SPREAD_SMALL] / 4;
    const long min_small = std::max<long>(64, 1024 / share), min_big = std::max<long>(4, 256 / share);
    const long small_waves = std::max<long>(64, std::min<long>(L->ntiles, std::max<long>(sw, min_small)));
    const int gs = (int)std::min<long>((small_waves + kSpreadWaves - 1) / kSpreadWaves, 4096);
    const int gb = (int)std::max<long>(
        1, std::min<long>(L->ntiles, std::max<long>(g->NV / g->lp[BL_IBM_SPREAD_BIG], min_big)));
    a.n_small = gs;
    blocks = (unsigned)(gs + gb);
    return a;
}

// Host state once a spreading is enqueued: its force field and flags trade
// places with the lattice's, so that the last collision's field stays
// readable (velocity staging) while the next one is formed.
void spread_swap(bl_ibm g)
{
    bl_lattice L = g->lat;
    if (L->flags_full) {  // the buffer leaving the lattice has every tile set
        g->alt_full = true;
        L->flags_full = false;
    }
    std::swap(L->tile_flags, g->flags_alt);  // this step's tiles carry the force now
    std::swap(L->force, g->force_alt);
    g->alt ^= 1;
    g->bins_dirty = false;
}

template <class S, class R>
void launch_spread_s(bl_ibm g, hipStream_t s)
{
    unsigned nb;
    const SpreadArgs<R> a = spread_args<R>(g, nb);
    if (g->S == 4) hipLaunchKernelGGL((k_spread<S, 4, R>), dim3(nb), dim3(256), 0, s, a);
    else if (g->S == 3) hipLaunchKernelGGL((k_spread<S, 3, R>), dim3(nb), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((k_spread<S, 2, R>), dim3(nb), dim3(256), 0, s, a);
}

int launch_spread(bl_ibm g, hipStream_t s)
{
    if (g->NV == 0) return BL_OK;
    int rc = vreal_matches_storage(g);
    if (rc) return rc;
    const int st = g->lat->storage;
    if (st == BL_STORE_F64) launch_spread_s<double, double>(g, s);
    else if (st == BL_STORE_F32) launch_spread_s<float, float>(g, s);
    else launch_spread_s<__half, float>(g, s);
    BL_CHECK_LAUNCH();
    spread_swap(g);
    return BL_OK;
}

// spreading | interpolation + advection, one launch: neither reads what the
// other writes
template <class S, class R>
void launch_spread_interp(bl_ibm g, hipStream_t s)
{
    unsigned nsp;
    const SpreadArgs<R> sp = spread_args<R>(g, nsp);
    spread_swap(g);
    const InterpArgs<R> ia = interp_args<R>(g, reset_next_of(g, s));
    const dim3 grid(nsp + interp_blocks(g));
    if (g->S == 4) hipLaunchKernelGGL((k_spread_interp<S, 4, R>), grid, dim3(256), 0, s, sp, (int)nsp, ia);
    else if (g->S == 3) hipLaunchKernelGGL((k_spread_interp<S, 3, R>), grid, dim3(256), 0, s, sp, (int)nsp, ia);
    else hipLaunchKernelGGL((k_spread_interp<S, 2, R>), grid, dim3(256), 0, s, sp, (int)nsp, ia);
}

int do_interpolate(bl_ibm g)
{
    int rc;
    if ((rc = do_bin(g, g->lat->stream))) return rc;
    if ((rc = launch_stage(g, g->lat->stream))) return rc;
    return launch_interp(g, false, g->lat->stream);
}

// Vertex forces on stream s: particle-particle forces into their own
// buffer, per-element membrane forces, then the per-vertex sum.
template <class R>
ElemArgs<R> elem_args(bl_ibm g)
{
    ElemArgs<R> a;
    a.f = force_view<R>(g);
    a.NT = g->NT;
    a.NP = g->NP;
    a.NL = g->NL;
    a.ec_pair = g->ec_pair;
    a.ec_link = g->ec_link;
    a.ec = (R*)g->ec;
    a.xcd = g->lp[BL_IBM_XCD];
    return a;
}

// `walls`: with the wall-interaction decorators and the particle-particle
// forces of this step (when there are any)
template <class R>
GatherArgs<R> gather_args(bl_ibm g, bool walls)
{
    GatherArgs<R> a;
    a.f = force_view<R>(g);
    a.NV = g->NV;
    a.ec_pair = g->ec_pair;
    a.ec_link = g->ec_link;
    a.ec = (const R*)g->ec;
    a.force = (R*)g->force;
    if (walls) a.deco = deco_set(g);
    else a.deco.n = 0;
    a.fpp = walls && !g->pp.empty() ? (const R*)g->pp_force : nullptr;
    a.ext = walls && g->has_ext ? (const R*)g->ext_force : nullptr;
    a.xcd = g->lp[BL_IBM_XCD];
    return a;
}

// per-element membrane forces, then the per-vertex sum (`walls`: with the
// decorators, particle-particle and host-given forces)
template <class R, int GL>
void launch_gather(bl_ibm g, hipStream_t s, bool walls)
{
    hipLaunchKernelGGL((k_vertex_gather<R, GL>), dim3(nblk(GL * g->NV)), dim3(256), 0, s, gather_args<R>(g, walls));
}

void launch_vertex_forces(bl_ibm g, hipStream_t s, bool walls)
{
    with_vreal(g, [&](auto tag) {
        using R = decltype(tag);
        const int gl = g->lp[BL_IBM_GATHER_LANES];
        if (gl == 2) launch_gather<R, 2>(g, s, walls);
        else if (gl == 8) launch_gather<R, 8>(g, s, walls);
        else launch_gather<R, 4>(g, s, walls);
        return 0;
    });
}

void launch_membrane(bl_ibm g, hipStream_t s, bool walls)
{
    const int eb = g->lp[BL_IBM_ELEM_BLOCK];
    with_vreal(g, [&](auto tag) {
        using R = decltype(tag);
        hipLaunchKernelGGL(k_elem_forces<R>, dim3(nblk(g->NT + g->NP + g->NL, eb)), dim3(eb), 0, s, elem_args<R>(g));
        return 0;
    });
    launch_vertex_forces(g, s, walls);
}

// binning | membrane element forces, one launch
int bin_elem_launch(bl_ibm g, hipStream_t s)
{
    int rc;
    if (!g->prepped && (rc = prep_bin(g, s))) return rc;
    g->prepped = false;
    with_vreal(g, [&](auto tag) {
        using R = decltype(tag);
        const int bb = g->lp[BL_IBM_BIN_BLOCK];  // both halves of the paired launch
        const int ne = (int)nblk(g->NT + g->NP + g->NL, bb);
        with_bin_form(g, bb, [&](auto form, int nb) {
            hipLaunchKernelGGL((k_bin_elem<R, decltype(form)::value>), dim3(nb + ne), dim3(bb), 0, s, bin_args<R>(g),
                               nb, elem_args<R>(g));
        });
        return 0;
    });
    BL_CHECK_LAUNCH();
    binned(g);
    return BL_OK;
}

int do_forces(bl_ibm g, hipStream_t s)
{
    int rc;
    const bool pp = !g->pp.empty() && g->NV;
    if (pp && (rc = interactions_launch(g, s))) return rc;
    if (g->NV) launch_membrane(g, s, true);
    BL_CHECK_LAUNCH();
    return BL_OK;
}

int do_spread(bl_ibm g)
{
    int rc;
    if (!g->binned && (rc = do_bin(g, g->lat->stream))) return rc;
    return launch_spread(g, g->lat->stream);
}

int do_move(bl_ibm g)
{
    hipStream_t s = g->lat->stream;
    if (g->NV)
        with_vreal(g, [&](auto tag) {
            using R = decltype(tag);
            hipLaunchKernelGGL(k_move<R>, dim3(nblk(3 * g->NV)), dim3(256), 0, s, g->NV, (R*)g->pos,
                               (const R*)g->vel);
            return 0;
        });
    BL_CHECK_LAUNCH();
    g->binned = false;
    return update_particles(g, 1);
}

int do_voxelize(bl_ibm g, hipStream_t s)
{
    bl_lattice L = g->lat;
    if (L->omega_c0 == L->omega_c1 || g->NT == 0) return BL_OK;
    const Grid gd = grid_of(L);
    with_vreal(g, [&](auto tag) {
        using R = decltype(tag);
        hipLaunchKernelGGL(k_ray_hits<R>, dim3(nblk(g->NT)), dim3(256), 0, s, force_view<R>(g), gd, g->NT, g->col_bits,
                           g->n_hits);
        return 0;
    });
    hipLaunchKernelGGL(k_fill_columns, dim3(nblk((long)L->nx * L->ny, kFillCols)), dim3(256), 0, s, gd, g->col_bits,
                       g->n_hits, g->hit_cap, g->n_active, g->phase);
    BL_CHECK_LAUNCH();
    if (L->phase != g->phase) {
        L->phase = g->phase;
        ++L->gen;
    }
    return BL_OK;
}

// Overflow flags accumulate on the device over any number of steps; this
// reads and clears them.
int check_overflow(bl_ibm g)
{
    int st[3] = {0, 0, 0};
    BL_HIP(hipMemcpyAsync(st, g->n_active, sizeof(st), hipMemcpyDeviceToHost, g->lat->stream));
    BL_HIP(hipStreamSynchronize(g->lat->stream));
    if (st[2]) {
        hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, g->lat->stream, g->n_active + 2, 1L, 0);
        BL_CHECK_LAUNCH();
    }
    if (st[2] & 1)
        return fail(BL_ERR_CAPACITY, "immersed boundary: more than " + std::to_string(kTileCap) +
                                         " stencils touch one 4x4x4 tile");
    if (st[2] & 2) return fail(BL_ERR_CAPACITY, "voxelization: more than 64 ray hits per triangle");
    if (st[2] & 4)
        return fail(BL_ERR_STATE, "immersed boundary: a vertex position is not finite (the membrane diverged)");
    return BL_OK;
}

// One IBM step, in one stream (with the stage timing events; spreading and
// interpolation are one of the timed stages and pair up: a 24^3 box 116 ->
// 111 us a step) ...
int step_serial(bl_ibm g)
{
    int rc;
    hipStream_t s = g->lat->stream;
    mark(g, 0);
    if ((rc = do_bin(g, s))) return rc;
    mark(g, 1);
    if ((rc = do_forces(g, s))) return rc;
    mark(g, 2);
    if ((rc = launch_stage(g, s))) return rc;
    if (use_pairs(g)) {
        if ((rc = vreal_matches_storage(g))) return rc;
        const int st = g->lat->storage;
        if (st == BL_STORE_F64) launch_spread_interp<double, double>(g, s);
        else if (st == BL_STORE_F32) launch_spread_interp<float, float>(g, s);
        else launch_spread_interp<__half, float>(g, s);
        BL_CHECK_LAUNCH();
    } else {
        if ((rc = launch_spread(g, s))) return rc;
        if ((rc = launch_interp(g, true, s, true))) return rc;
    }
    mark(g, 3);
    g->binned = false;
    if ((rc = update_particles(g, 1, s))) return rc;
    mark(g, 4);
    if ((rc = do_voxelize(g, s))) return rc;
    mark(g, 5);
    return BL_OK;
}

// ... or forked over the lattice stream M and the boundary's stream A, so
// that independent stages overlap:
//   A: particle-particle forces (when there are any) and membrane forces
//      (read the positions before the move); after the binning, spreading
//      into the second force buffer (it needs the lists and the forces,
//      not the staging)
//   M: binning, velocity staging (the last collision's force field and the
//      new tile flags), then, once the forces have read the positions,
//      interpolation + advection (the launch also readies the next
//      binning's list: the flags and list two steps back are free once
//      staged), geometry, voxelization; then joins A (the collision reads
//      the spread force field).
// The chain that ends at the collision stays on one queue; only the start
// of A, the binning's lists and the spread field cross between queues.
int step_forked(bl_ibm g)
{
    int rc;
    hipStream_t M = g->lat->stream, A = g->aux[0];
    hipEvent_t* e = g->fev;
    BL_HIP(hipEventRecord(e[0], M));
    BL_HIP(hipStreamWaitEvent(A, e[0], 0));
    if ((rc = do_forces(g, A))) return rc;
    BL_HIP(hipEventRecord(e[1], A));
    if ((rc = do_bin(g, M, e[2]))) return rc;
    if ((rc = launch_stage(g, M))) return rc;
    BL_HIP(hipStreamWaitEvent(A, e[2], 0));
    if ((rc = launch_spread(g, A))) return rc;
    BL_HIP(hipEventRecord(e[4], A));
    BL_HIP(hipStreamWaitEvent(M, e[1], 0));
    if ((rc = launch_interp(g, true, M, true))) return rc;
    g->binned = false;
    if ((rc = update_particles(g, 1, M))) return rc;
    if ((rc = do_voxelize(g, M))) return rc;
    BL_HIP(hipStreamWaitEvent(M, e[4], 0));
    return BL_OK;
}

// Whether coupled steps carry the velocity staging in the collision
// (step_fused).  Only without a phase field: the collision of a step reads
// the phase voxelized from the moved vertices, which need the staged
// velocity first.  By default for kPairedVertices vertices or more ...
bool fused_large(bl_ibm g)
{
    bl_lattice L = g->lat;
    if (g->fused_staging == 0 || g->NV == 0 || L->omega_c0 != L->omega_c1) return false;
    return g->fused_staging == 1 || g->NV >= kPairedVertices;
}

// ... and, outside batches of boxes, for fewer where most tiles of a lattice
// of kStagedBytes of populations are staged: the pass that the collision
// saves reads them all again (171 x 70 x 101 FP64, 184 MB: 39 us beside the
// gather, 10 more in the collision; 223 -> 213 us a step), and the two stages
// it would have shared launches with cost about 15 us by themselves, what
// the pass takes over some 70 MB.
constexpr size_t kStagedBytes = 96u << 20;
bool use_fused(bl_ibm g)
{
    bl_lattice L = g->lat;
    if (fused_large(g)) return true;
    return g->fused_staging < 0 && g->layered < 0 && g->NV > 0 && L->omega_c0 == L->omega_c1 && spread_dense(g) &&
           (size_t)Q * L->stride * L->pop_bytes >= kStagedBytes;
}

// One coupled step with the velocity staging carried by the collision.
// The reference's order (computeVelocity, interpolate, spread, move,
// collide) has the collision depend only on the spread force, and the
// interpolation only on the staged velocity, so the step runs as
//   A: particle-particle and membrane forces (positions before the move)
//   M: binning; then, after A, spreading; collide-and-stream, which also
//      stages u (pre-collision populations, the last collision's force
//      field) on the touched tiles; post-stream walls; interpolation +
//      advection (readying the next binning's list); geometry.
// (With few vertices A is on M too, the element forces in the binning's
// launch.)
// The staged values are those of k_stage_u; one pass over the touched
// populations is saved.
int step_fused(bl_ibm g)
{
    int rc;
    bl_lattice L = g->lat;
    hipStream_t M = L->stream, A = g->aux[0];
    hipEvent_t* e = g->fev;
    if (use_pairs(g)) {
        if (!g->pp.empty() && (rc = interactions_launch(g, M))) return rc;
        if ((rc = bin_elem_launch(g, M))) return rc;
        launch_vertex_forces(g, M, true);
    } else {
        BL_HIP(hipEventRecord(e[0], M));
        BL_HIP(hipStreamWaitEvent(A, e[0], 0));
        if ((rc = do_forces(g, A))) return rc;
        BL_HIP(hipEventRecord(e[1], A));
        if ((rc = do_bin(g, M))) return rc;
        BL_HIP(hipStreamWaitEvent(M, e[1], 0));
    }
    if ((rc = launch_spread(g, M))) return rc;
    // after the swap: the lattice holds this step's field and flags (the
    // touched tiles), the boundary's spare buffers the last collision's
    L->emit_u = g->ut;
    L->emit_force = g->force_alt;
    L->emit_flags = g->flags_alt;
    rc = collide_stream_launch(L);
    L->emit_u = nullptr;
    L->emit_force = nullptr;
    L->emit_flags = nullptr;
    if (rc) return rc;
    if ((rc = velocity_walls_launch(L))) return rc;
    if ((rc = launch_interp(g, true, M, true))) return rc;
    g->binned = false;
    return update_particles(g, 1, M);
}

// One coupled step on the lattice stream alone, as four launches before
// the collision, each pairing two stages that do not read each other's
// output:
//   binning | membrane element forces (both read the positions only)
//   vertex force gather | velocity staging (the binning's tiles, the last
//     collision's field and flags)
//   spreading | interpolation + advection (the launch also readies the
//     next binning's list)
//   geometry (then voxelization, with a phase field)
// The reference's order and every value are those of the other layouts;
// no stage waits on another queue.
// force gather (GL lanes per vertex) | velocity staging, one launch
template <class S, bool EITHER, class R, int GL>
void launch_gather_stage_of(bl_ibm g, hipStream_t s)
{
    const int ng = (int)nblk(GL * g->NV);
    const StageArgs sa = stage_args(g);
    const dim3 g2(ng + stage_blocks(g, sa.active != nullptr));
    if (g->lat->steps & 1)
        hipLaunchKernelGGL((k_gather_stage<S, true, EITHER, R, GL>), g2, dim3(256), 0, s, gather_args<R>(g, true), ng, sa);
    else
        hipLaunchKernelGGL((k_gather_stage<S, false, EITHER, R, GL>), g2, dim3(256), 0, s, gather_args<R>(g, true), ng, sa);
}

// From 2^20 cells on by a kernel that has no list form: with it the cells'
// form holds more registers, and 256 x 128 x 128 with 96 cells, FP16s, odd |
// even steps, took 39.5 | 30.8 us, without 34.9 | 27.4.  Below, the kernel
// with both is the shorter one (64^3 FP64 5.1 | 4.9 us, without 5.5 | 5.2).
// k_stage_u, alone on its stream, keeps both: the membrane's kernels beside
// it lose more to the cells' higher occupancy than it gains (256 x 128 x 128
// FP64 with 256 800 vertices and a phase field: 676 us a coupled step, 707
// without).
template <class S, class R, int GL>
void launch_gather_stage(bl_ibm g, hipStream_t s)
{
    if (g->lat->ncell >= 1l << 20 && !stage_by_list(g)) launch_gather_stage_of<S, false, R, GL>(g, s);
    else launch_gather_stage_of<S, true, R, GL>(g, s);
}

template <class S>
int step_layered_s(bl_ibm g)
{
    using R = typename VRof<S>::T;
    int rc;
    bl_lattice L = g->lat;
    if ((rc = vreal_matches_storage(g))) return rc;
    hipStream_t s = L->stream;
    if (!g->pp.empty() && (rc = interactions_launch(g, s))) return rc;
    if ((rc = bin_elem_launch(g, s))) return rc;
    const int gl = g->lp[BL_IBM_GATHER_LANES];
    if (gl == 2) launch_gather_stage<S, R, 2>(g, s);
    else if (gl == 8) launch_gather_stage<S, R, 8>(g, s);
    else launch_gather_stage<S, R, 4>(g, s);
    launch_spread_interp<S, R>(g, s);
    BL_CHECK_LAUNCH();
    g->binned = false;
    if ((rc = update_particles(g, 1, s))) return rc;
    return do_voxelize(g, s);
}

int step_layered(bl_ibm g)
{
    const int st = g->lat->storage;
    if (st == BL_STORE_F64) return step_layered_s<double>(g);
    if (st == BL_STORE_F32) return step_layered_s<float>(g);
    return step_layered_s<__half>(g);
}

// Whether coupled steps without fused staging run as step_layered (one
// stream) rather than step_forked (two): by default below 65 536 vertices,
// where the stages are a few workgroups each and a wait across queues
// costs more than the overlap gains.
bool use_layered(bl_ibm g)
{
    if (g->NV == 0 || g->layered == 0) return false;
    return g->layered == 1 || use_pairs(g);
}

// n coupled steps enqueued on the lattice stream
int steps_forked(bl_ibm g, int n)
{
    int rc;
    for (int k = 0; k < n; ++k) {
        if (use_fused(g)) {
            if ((rc = step_fused(g))) return rc;
            continue;
        }
        if ((rc = use_layered(g) ? step_layered(g) : step_forked(g))) return rc;
        if ((rc = collide_stream_launch(g->lat))) return rc;
        if ((rc = velocity_walls_launch(g->lat))) return rc;
    }
    return BL_OK;
}

// ------------------------------------------------ batches of boxes
// An ensemble of independent boxes whose steps all take the paired-stage
// layout (step_layered) runs each stage as one launch over every box:
// LayeredEntry holds one box's arguments of one step, as step_layered
// forms them; a batched kernel finds its box with batch_box over the
// launch's per-box workgroup offsets and runs the box-local workgroup with
// that box's arguments.  plan_layered advances the boundary's host state
// exactly as step_layered does, without launching.
template <class R>
struct LayeredEntry {
    ListReset reset;
    int nr;  // workgroups of the binning's list reset (0: the list is ready)
    BinArgs<R> bin;
    ElemArgs<R> elem;
    int nb, ne;
    GatherArgs<R> gather;
    StageArgs stage;
    int ng, nst;
    SpreadArgs<R> spread;
    InterpArgs<R> interp;
    int nsp, nip;
    GeomArgs<R> geom;
};

// Whether a boundary's coupled step can join a batch: the paired-stage
// layout, no particle-particle forces or phase field, no pending clear of
// its tile buffers, and the vertex type of its storage.
bool layered_batchable(bl_ibm g)
{
    const bl_lattice L = g->lat;
    return L && g->inited && g->NV > 0 && use_layered(g) && !fused_large(g) && g->pp.empty() &&
           L->omega_c0 == L->omega_c1 && !g->bins_dirty && !g->alt_full && !ibm_needs_settle(g) && !g->timing &&
           g->n_rigid == 0 && g->vreal == (L->storage == BL_STORE_F64 ? 8 : 4);
}

// One step's entry; BL_ERR_STATE when a clear of the tile buffers would be
// needed in the middle of the step (the batch is then not used).
template <class R>
int plan_layered(bl_ibm g, LayeredEntry<R>& E, int share)
{
    bl_lattice L = g->lat;
    E.nr = 0;
    if (!g->prepped) {
        if (g->bins_dirty || g->alt_full) return BL_ERR_STATE;
        E.reset = list_reset_of(g);
        E.nr = (int)std::min<long>(nblk(L->ntiles), kResetBlocks);
        g->prepped = true;
    }
    g->prepped = false;
    E.bin = bin_args<R>(g);
    E.elem = elem_args<R>(g);
    E.nb = bin_blocks(g, 256, false);
    E.ne = (int)nblk(g->NT + g->NP + g->NL);
    binned(g);
    E.gather = gather_args<R>(g, true);
    E.stage = stage_args(g);
    E.ng = (int)nblk((long)g->lp[BL_IBM_GATHER_LANES] * g->NV);
    E.nst = (int)stage_blocks(g, false);  // a batch stages by cells
    unsigned nsp;
    E.spread = spread_args<R>(g, nsp, share);
    E.nsp = (int)nsp;
    spread_swap(g);
    if (g->bins_dirty || g->alt_full) return BL_ERR_STATE;
    g->prepped = true;
    E.interp = interp_args<R>(g, list_reset_of(g));
    E.nip = (int)interp_blocks(g);
    g->binned = false;
    E.geom = geom_args<R>(g, 1);
    return BL_OK;
}

template <class R>
__global__ void __launch_bounds__(256) k_reset_batch(const LayeredEntry<R>* __restrict__ tab,
                                                     const int* __restrict__ base, int nbox)
{
    const int box = batch_box(base, nbox, (int)blockIdx.x);
    const LayeredEntry<R>& E = tab[box];
    list_reset(E.reset, (int)blockIdx.x - base[box], E.nr);
}

template <class R>
__global__ void __launch_bounds__(256) k_bin_elem_batch(const LayeredEntry<R>* __restrict__ tab,
                                                        const int* __restrict__ base, int nbox)
{
    const int box = batch_box(base, nbox, (int)blockIdx.x);
    const LayeredEntry<R>& E = tab[box];
    const int bx = (int)blockIdx.x - base[box];
    if (bx < E.nb) bin_group<R, BIN_ONE>(ibm_block(bx, E.nb, E.bin.xcd), E.bin);
    else elem_body<R>(ibm_block(bx - E.nb, E.ne, E.elem.xcd), E.elem);
}

template <class S, bool SWAPPED, class R, int GL>
__global__ void __launch_bounds__(256) k_gather_stage_batch(const LayeredEntry<R>* __restrict__ tab,
                                                            const int* __restrict__ base, int nbox)
{
    const int box = batch_box(base, nbox, (int)blockIdx.x);
    const LayeredEntry<R>& E = tab[box];
    const int bx = (int)blockIdx.x - base[box];
    if (bx < E.ng) gather_body<R, GL>(ibm_block(bx, E.ng, E.gather.xcd), E.gather);
    else stage_body<S, SWAPPED, false>(bx - E.ng, E.nst, E.stage);
}

template <class S, int SW, class R>
__global__ void __launch_bounds__(256) k_spread_interp_batch(const LayeredEntry<R>* __restrict__ tab,
                                                             const int* __restrict__ base, int nbox)
{
    const int box = batch_box(base, nbox, (int)blockIdx.x);
    const LayeredEntry<R>& E = tab[box];
    const int bx = (int)blockIdx.x - base[box];
    if (bx < E.nsp) spread_body<S, SW, R>(bx, E.nsp, E.spread);
    else interp_body<typename Pop<S>::C, SW, true, R>(bx - E.nsp, E.nip, E.interp);
}

// The interpolation with advection alone (batches whose velocity staging
// rides on the collision: it runs after the collide-and-stream).
template <class S, int SW, class R>
__global__ void __launch_bounds__(256) k_interp_batch(const LayeredEntry<R>* __restrict__ tab,
                                                      const int* __restrict__ base, int nbox)
{
    const int box = batch_box(base, nbox, (int)blockIdx.x);
    const LayeredEntry<R>& E = tab[box];
    interp_body<typename Pop<S>::C, SW, true, R>((int)blockIdx.x - base[box], E.nip, E.interp);
}

template <class R>
__global__ void __launch_bounds__(256) k_geom_partial_batch(const LayeredEntry<R>* __restrict__ tab,
                                                            const int* __restrict__ base, int nbox)
{
    const int box = batch_box(base, nbox, (int)blockIdx.x);
    geom_partial_body<R>((int)blockIdx.x - base[box], tab[box].geom);
}

template <class R>
__global__ void __launch_bounds__(64) k_geom_final_batch(const LayeredEntry<R>* __restrict__ tab,
                                                         const int* __restrict__ base, int nbox)
{
    const int box = batch_box(base, nbox, (int)blockIdx.x);
    geom_final_body<R>((int)blockIdx.x - base[box], tab[box].geom);
}

template <class R>
__global__ void __launch_bounds__(kGeomBlock) k_geom_batch(const LayeredEntry<R>* __restrict__ tab,
                                                           const int* __restrict__ base, int nbox)
{
    const int box = batch_box(base, nbox, (int)blockIdx.x);
    geom_body<R>((int)blockIdx.x - base[box], tab[box].geom);
}

}  // namespace

// Two coupled steps of every box of an ensemble as batched launches: the
// entries and workgroup offsets of every launch in one device buffer.
struct EnsembleBatch {
    int storage = 0, sw = 4, gl = 4;
    int order[2] = {0, 0};  // collide workgroup order per AA parity (collide_block modes)
    int nt[2] = {0, 0};     // and nontemporal level
    bool any_ibm = false;
    // velocity staging carried by the batched collision (every box has an
    // immersed boundary): no staging pass, the interpolation after the
    // collide-and-stream and the walls, as a single box's fused step
    bool fused = false;
    void* dev = nullptr;  // entries and offsets of both steps
    struct Launch {
        size_t tab = 0, base = 0;  // byte offsets into dev
        int nbox = 0;
        unsigned nblk = 0;
    };
    struct Step {
        bool swapped = false;  // the IBM stages' AA parity (before the collision)
        Launch reset, bin_elem, gather_stage, spread_interp, interp, geom_partial, geom_final, geom, collide, vwall;
        CollidePlan c0;        // template choices of the collide launch
        bool vw_swapped = false;
    } step[2];
};

namespace {

// Appends n objects to a host byte image (8-byte aligned), returning their offset.
template <class T>
size_t put(std::vector<char>& img, const T* p, size_t n)
{
    size_t off = (img.size() + 15) & ~(size_t)15;
    img.resize(off + sizeof(T) * n);
    if (n) memcpy(img.data() + off, p, sizeof(T) * n);
    return off;
}

// the workgroup offsets of a launch over boxes with the given counts
EnsembleBatch::Launch put_launch(std::vector<char>& img, size_t tab, const std::vector<int>& counts)
{
    EnsembleBatch::Launch l;
    std::vector<int> base(counts.size() + 1, 0);
    for (size_t k = 0; k < counts.size(); ++k) base[k + 1] = base[k] + counts[k];
    l.tab = tab;
    l.base = put(img, base.data(), base.size());
    l.nbox = (int)counts.size();
    l.nblk = (unsigned)base.back();
    return l;
}

template <class R>
int batch_plan_ibm(const std::vector<bl_ibm>& gs, std::vector<char>& img, EnsembleBatch::Step& st, bool fused,
                   std::vector<LatView>* emit)
{
    std::vector<LayeredEntry<R>> E(gs.size());
    for (size_t k = 0; k < gs.size(); ++k) {
        const int rc = plan_layered<R>(gs[k], E[k], (int)gs.size());
        if (rc) return rc;
        if (fused) {
            // after the step's spread swap: the boundary's spare field and
            // flags are the last collision's (what the staging reads)
            LatView& v = (*emit)[k];
            v.emit_u = gs[k]->ut;
            v.emit_force = gs[k]->force_alt;
            v.emit_flags = gs[k]->flags_alt;
        }
    }
    const size_t tab = put(img, E.data(), E.size());
    std::vector<int> nr, nbe, ngs, nsi, nip, nch, npa, ngo;
    for (size_t k = 0; k < gs.size(); ++k) {
        nr.push_back(E[k].nr);
        nbe.push_back(E[k].nb + E[k].ne);
        // fused: the gather alone and the spreading alone (every workgroup
        // index stays below the first stage's count)
        ngs.push_back(E[k].ng + (fused ? 0 : E[k].nst));
        nsi.push_back(E[k].nsp + (fused ? 0 : E[k].nip));
        nip.push_back(fused ? E[k].nip : 0);
        nch.push_back(gs[k]->geom_one ? 0 : gs[k]->nchunk);
        npa.push_back(gs[k]->geom_one ? 0 : gs[k]->np);
        ngo.push_back(gs[k]->geom_one ? gs[k]->np : 0);
    }
    st.reset = put_launch(img, tab, nr);
    st.bin_elem = put_launch(img, tab, nbe);
    st.gather_stage = put_launch(img, tab, ngs);
    st.spread_interp = put_launch(img, tab, nsi);
    st.interp = put_launch(img, tab, nip);
    st.geom_partial = put_launch(img, tab, nch);
    st.geom_final = put_launch(img, tab, npa);
    st.geom = put_launch(img, tab, ngo);
    return BL_OK;
}

// The immersed-boundary launches of one batched step: before the collision
// (after = false) the binning with element forces, the gather (with the
// staging unless fused) and the spreading (with the interpolation unless
// fused), then the geometry unless fused; after the collision and the
// walls (after = true, fused only) the interpolation and the geometry.
template <class S>
void batch_launch_ibm(const EnsembleBatch& B, const EnsembleBatch::Step& st, bool after, hipStream_t s)
{
    using R = typename VRof<S>::T;
    const char* d = (const char*)B.dev;
    auto tab = [&](const EnsembleBatch::Launch& l) { return (const LayeredEntry<R>*)(d + l.tab); };
    auto base = [&](const EnsembleBatch::Launch& l) { return (const int*)(d + l.base); };
    auto go = [&](auto kern, const EnsembleBatch::Launch& l, int blk) {
        if (l.nblk) hipLaunchKernelGGL(kern, dim3(l.nblk), dim3(blk), 0, s, tab(l), base(l), l.nbox);
    };
    if (!after) {
        go(k_reset_batch<R>, st.reset, 256);
        go(k_bin_elem_batch<R>, st.bin_elem, 256);
        auto gs = [&](auto sw_tag) {
            constexpr bool SWP = decltype(sw_tag)::value;
            if (B.gl == 2) go(k_gather_stage_batch<S, SWP, R, 2>, st.gather_stage, 256);
            else if (B.gl == 8) go(k_gather_stage_batch<S, SWP, R, 8>, st.gather_stage, 256);
            else go(k_gather_stage_batch<S, SWP, R, 4>, st.gather_stage, 256);
        };
        if (st.swapped) gs(std::true_type{});
        else gs(std::false_type{});
        if (B.sw == 4) go(k_spread_interp_batch<S, 4, R>, st.spread_interp, 256);
        else if (B.sw == 3) go(k_spread_interp_batch<S, 3, R>, st.spread_interp, 256);
        else go(k_spread_interp_batch<S, 2, R>, st.spread_interp, 256);
        if (B.fused) return;
    } else {
        if (B.sw == 4) go(k_interp_batch<S, 4, R>, st.interp, 256);
        else if (B.sw == 3) go(k_interp_batch<S, 3, R>, st.interp, 256);
        else go(k_interp_batch<S, 2, R>, st.interp, 256);
    }
    go(k_geom_partial_batch<R>, st.geom_partial, 256);
    go(k_geom_final_batch<R>, st.geom_final, 64);
    go(k_geom_batch<R>, st.geom, kGeomBlock);
}

}  // namespace

int ensemble_batch_build(const std::vector<bl_lattice>& lats, const std::vector<bl_ibm>& ibms, const int order[2],
                         const int nt[2], EnsembleBatch** out)
{
    *out = nullptr;
    const size_t n = lats.size();
    if (n < 2) return BL_OK;
    std::vector<bl_ibm> gs;
    int sw = 0, gl = 0;
    for (size_t k = 0; k < n; ++k) {
        const bl_lattice L = lats[k];
        if (!L->guo.empty() || L->storage != lats[0]->storage || (L->steps & 1) != (lats[0]->steps & 1)) return BL_OK;
        if (!collide_batchable(collide_plan(L), collide_plan(lats[0]))) return BL_OK;
        const bl_ibm g = ibms[k];
        if (!g) continue;
        if (!layered_batchable(g)) return BL_OK;
        if ((sw && g->S != sw) || (gl && g->lp[BL_IBM_GATHER_LANES] != gl)) return BL_OK;
        sw = g->S;
        gl = g->lp[BL_IBM_GATHER_LANES];
        gs.push_back(g);
    }
    // plan both steps; the host state of every box advances two steps and
    // its step count is put back afterwards (nothing has run)
    std::vector<long long> s0(n);
    for (size_t k = 0; k < n; ++k) s0[k] = lats[k]->steps;
    EnsembleBatch* B = new EnsembleBatch();
    B->storage = lats[0]->storage;
    B->sw = sw ? sw : 4;
    B->gl = gl ? gl : 4;
    B->any_ibm = !gs.empty();
    B->fused = gs.size() == n && collide_plan(lats[0]).fm == 2;
    B->order[0] = order[0];
    B->order[1] = order[1];
    B->nt[0] = nt[0];
    B->nt[1] = nt[1];
    std::vector<char> img;
    int rc = BL_OK;
    for (int k = 0; k < 2 && rc == BL_OK; ++k) {
        EnsembleBatch::Step& st = B->step[k];
        st.swapped = (lats[0]->steps & 1) != 0;
        // the collide views after the boundaries' plans (their spread swap
        // hands each lattice this step's force field), with the staging
        // pointers the plans recorded when fused
        std::vector<LatView> emit(n);
        if (!gs.empty()) {
            if (B->storage == BL_STORE_F64) rc = batch_plan_ibm<double>(gs, img, st, B->fused, &emit);
            else rc = batch_plan_ibm<float>(gs, img, st, B->fused, &emit);
            if (rc) break;
        }
        std::vector<LatView> views;
        std::vector<int> cnt;
        st.c0 = collide_plan(lats[0]);
        for (size_t k = 0; k < n; ++k) {
            const bl_lattice L = lats[k];
            LatView v = collide_plan(L).v;
            if (B->fused) {
                v.emit_u = emit[k].emit_u;
                v.emit_force = emit[k].emit_force;
                v.emit_flags = emit[k].emit_flags;
            }
            views.push_back(v);
            cnt.push_back((int)((L->ncell + 255) / 256));
            collide_commit(L);
        }
        st.collide = put_launch(img, put(img, views.data(), views.size()), cnt);
        std::vector<VwallPlan> vw;
        std::vector<int> vcnt;
        st.vw_swapped = (lats[0]->steps & 1) != 0;
        for (bl_lattice L : lats)
            if (L->has_vwall && L->mask) {
                vw.push_back(VwallPlan{view_of(L), L->nwall});
                vcnt.push_back(vwall_blocks(L));
            }
        const size_t vtab = put(img, vw.data(), vw.size());
        st.vwall = put_launch(img, vtab, vcnt);
    }
    for (size_t k = 0; k < n; ++k) lats[k]->steps = s0[k];
    if (rc) {  // a clear was due mid-step: the ensemble uses per-box branches
        delete B;
        return rc == BL_ERR_STATE ? BL_OK : rc;
    }
    if (hipMalloc(&B->dev, img.size()) != hipSuccess ||
        hipMemcpy(B->dev, img.data(), img.size(), hipMemcpyHostToDevice) != hipSuccess) {
        hipFree(B->dev);
        delete B;
        return fail(BL_ERR_HIP, "ensemble batch: device tables");
    }
    *out = B;
    return BL_OK;
}

int ensemble_batch_launch(const EnsembleBatch* B, hipStream_t s)
{
    const char* d = (const char*)B->dev;
    for (int k = 0; k < 2; ++k) {
        const EnsembleBatch::Step& st = B->step[k];
        auto ibm = [&](bool after) {
            if (B->storage == BL_STORE_F64) batch_launch_ibm<double>(*B, st, after, s);
            else if (B->storage == BL_STORE_F32) batch_launch_ibm<float>(*B, st, after, s);
            else batch_launch_ibm<__half>(*B, st, after, s);
        };
        if (B->any_ibm) {
            ibm(false);
            BL_CHECK_LAUNCH();
        }
        int rc = collide_batch_launch(st.c0, B->fused, (const LatView*)(d + st.collide.tab),
                                      (const int*)(d + st.collide.base), st.collide.nbox, st.collide.nblk,
                                      B->order[st.c0.odd ? 1 : 0], B->nt[st.c0.odd ? 1 : 0], s);
        if (rc) return rc;
        if (st.vwall.nblk &&
            (rc = vwall_batch_launch(B->storage, st.vw_swapped, (const VwallPlan*)(d + st.vwall.tab),
                                     (const int*)(d + st.vwall.base), st.vwall.nbox, st.vwall.nblk, s)))
            return rc;
        if (B->fused) {
            ibm(true);
            BL_CHECK_LAUNCH();
        }
    }
    return BL_OK;
}

void ensemble_batch_free(EnsembleBatch* B)
{
    if (!B) return;
    hipFree(B->dev);
    delete B;
}

int ibm_step_launch(bl_ibm g, bool forked)
{
    int rc;
    if (forked) return steps_forked(g, 1);
    // on the lattice stream alone: paired stages unless stage times are taken
    if ((rc = !g->timing && use_layered(g) ? step_layered(g) : step_serial(g))) return rc;
    if ((rc = collide_stream_launch(g->lat))) return rc;
    return velocity_walls_launch(g->lat);
}

int ibm_check_overflow(bl_ibm g) { return check_overflow(g); }

void ibm_detach(bl_ibm g)
{
    for (auto& st : g->aux)
        if (st) hipStreamSynchronize(st);
    g->lat = nullptr;
}

int vreal_upload(bl_ibm g, void* dst, long off, const double* src, long n, hipStream_t s)
{
    if (n <= 0) return BL_OK;
    if (g->vreal == 8) {
        BL_HIP(hipMemcpyAsync((double*)dst + off, src, sizeof(double) * n, hipMemcpyHostToDevice, s));
        BL_HIP(hipStreamSynchronize(s));
        return BL_OK;
    }
    std::vector<float> tmp(src, src + n);
    BL_HIP(hipMemcpyAsync((float*)dst + off, tmp.data(), sizeof(float) * n, hipMemcpyHostToDevice, s));
    BL_HIP(hipStreamSynchronize(s));
    return BL_OK;
}

int vreal_download(bl_ibm g, double* dst, const void* src, long off, long n, hipStream_t s)
{
    if (n <= 0) return BL_OK;
    if (g->vreal == 8) {
        BL_HIP(hipMemcpyAsync(dst, (const double*)src + off, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        BL_HIP(hipStreamSynchronize(s));
        return BL_OK;
    }
    std::vector<float> tmp(n);
    BL_HIP(hipMemcpyAsync(tmp.data(), (const float*)src + off, sizeof(float) * n, hipMemcpyDeviceToHost, s));
    BL_HIP(hipStreamSynchronize(s));
    for (long i = 0; i < n; ++i) dst[i] = (double)tmp[i];
    return BL_OK;
}

void ibm_invalidate_graphs(bl_ibm g)
{
    g->graph_parity[0] = g->graph_parity[1] = -1;
    ++g->gen;
}

// Steps run eagerly while a loaded full force field is consumed, and for the
// first step after the body force changed (its velocity staging reads the
// previous body force; a captured step would bake that value in).
bool ibm_needs_settle(bl_ibm g)
{
    const bl_lattice L = g->lat;
    if (!L) return false;
    const bool g_changed = L->g_last[0] != L->g[0] || L->g_last[1] != L->g[1] || L->g_last[2] != L->g[2];
    return L->flags_full || g->alt_full || g_changed;
}

// The stages that place delta-kernel stencils on the lattice (binning,
// interpolation, spreading) need every periodic extent to hold one stencil
// width, so that a stencil never covers a cell twice; the membrane and
// collision-handler forces do not.
int need_stencil(bl_ibm g)
{
    int rc = need_init(g);
    if (rc) return rc;
    if ((rc = rigid_refuse_coupling(g))) return rc;
    const bl_lattice L = g->lat;
    const int n3[3] = {L->nx, L->ny, L->nz};
    for (int d = 0; d < 3; ++d)
        if (L->periodic[d] && n3[d] < 4)
            return fail(BL_ERR_ARG, "immersed boundary: the kernel stages need periodic extents of at least 4 "
                                    "(one stencil width)");
    return BL_OK;
}

}  // namespace bl

using namespace bl;

extern "C" {

int bl_ibm_create(bl_lattice lat, int kernel, bl_ibm* out)
{
    if (!lat || !out) return fail(BL_ERR_ARG, "bl_ibm_create: null argument");
    if (kernel < BL_KERNEL_ROMA || kernel > BL_KERNEL_TOPHAT) return fail(BL_ERR_ARG, "bl_ibm_create: unknown kernel");
    if (lat->ibm) return fail(BL_ERR_STATE, "bl_ibm_create: lattice already has an immersed boundary");
    bl_ibm g = new bl_ibm_s();
    g->lat = lat;
    g->kernel = kernel;
    g->S = kernel == BL_KERNEL_ROMA ? 3 : (kernel == BL_KERNEL_PESKIN ? 4 : 2);
    g->h = kernel == BL_KERNEL_ROMA ? 1.5 : (kernel == BL_KERNEL_PESKIN ? 2.0 : 1.0);
    lat->ibm = g;
    *out = g;
    return BL_OK;
}

int bl_ibm_destroy(bl_ibm g)
{
    if (!g) return BL_OK;
    if (g->lat) {
        hipStreamSynchronize(g->lat->stream);
        if (g->lat->phase == g->phase) g->lat->phase = g->lat->own_phase;
        g->lat->ibm = nullptr;
        ++g->lat->gen;
    }
    void* ptrs[] = {g->s_voff, g->s_toff, g->s_loff, g->s_poff, g->s_vtoff, g->s_vloff, g->s_vpoff, g->s_tri,
                    g->s_tri_area0, g->s_tri_geo0, g->s_rest, g->s_link, g->s_link_len, g->s_pair, g->s_pair_cs0,
                    g->s_vt_head, g->s_vt, g->s_vl_head, g->s_vl, g->s_vp_head, g->s_vp, g->s_area0, g->p_shape,
                    g->p_model, g->p_bug, g->p_params, g->p_voff, g->p_toff, g->p_loff, g->p_poff, g->p_geom,
                    g->p_delta, g->pos, g->vel, g->force, g->ec, g->ut, g->v_pos0,
                    g->tile_count, g->tile_list, g->active, g->n_active,
                    g->col_bits, g->n_hits, g->phase,
                    g->flags_alt, g->force_alt, g->p_choff, g->ch_partial, g->ch_tab, g->t_vert, g->v_inc, g->v_near, g->v_blend, g->v_part, g->t_part, g->r_part,
                    g->l_part, g->ext_force, g->r_state};
    for (void* p : ptrs) hipFree(p);
    interactions_free(g);
    for (auto& e : g->ev)
        if (e) hipEventDestroy(e);
    for (auto& e : g->fev)
        if (e) hipEventDestroy(e);
    for (auto& st : g->aux)
        if (st) {
            hipStreamSynchronize(st);
            hipStreamDestroy(st);
        }
    for (auto& ge : g->graph)
        if (ge) hipGraphExecDestroy(ge);
    delete g;
    return BL_OK;
}

int bl_shape_add(bl_ibm g, int nv, int nt, const double* rest_pos, const int* tri, int* shape_id)
{
    if (!g || !rest_pos || !tri || nv < 3 || nt < 1) return fail(BL_ERR_ARG, "bl_shape_add: bad argument");
    if (g->inited) return fail(BL_ERR_STATE, "bl_shape_add: shapes must be added before bl_ibm_init");
    ShapeHost sh;
    std::string err;
    if (!build_shape(nv, nt, rest_pos, tri, sh, &err)) return fail(BL_ERR_ARG, "bl_shape_add: " + err);
    g->shapes.push_back(std::move(sh));
    if (shape_id) *shape_id = (int)g->shapes.size() - 1;
    return BL_OK;
}

int bl_shape_info(bl_ibm g, int shape_id, double out[6])
{
    if (!g || !out || shape_id < 0 || shape_id >= (int)g->shapes.size()) return fail(BL_ERR_ARG, "bl_shape_info: bad argument");
    const ShapeHost& s = g->shapes[shape_id];
    out[0] = s.area;
    out[1] = s.volume;
    for (int d = 0; d < 3; ++d) out[2 + d] = s.center[d];
    out[5] = s.radius;
    return BL_OK;
}

int bl_particle_add(bl_ibm g, int shape_id, int model, const double* params, int nparams, const double* pos,
                    int bug_compatible, int* pid)
{
    if (!g || !params || !pos) return fail(BL_ERR_ARG, "bl_particle_add: null argument");
    if (g->inited) return fail(BL_ERR_STATE, "bl_particle_add: particles must be added before bl_ibm_init");
    if (shape_id < 0 || shape_id >= (int)g->shapes.size()) return fail(BL_ERR_ARG, "bl_particle_add: unknown shape");
    if (model < 0 || model > 3) return fail(BL_ERR_ARG, "bl_particle_add: unknown model");
    const int need = model <= 1 ? 2 : 7;
    if (nparams < need || nparams > 8) return fail(BL_ERR_ARG, "bl_particle_add: wrong number of parameters");
    bl_ibm_s::PartHost p;
    p.shape = shape_id;
    p.model = model;
    p.bug = bug_compatible ? 1 : 0;
    for (int k = 0; k < nparams; ++k) p.params[k] = params[k];
    if ((model == BL_MODEL_RBC || model == 3) && !(p.params[5] > 0))
        return fail(BL_ERR_ARG, "bl_particle_add: vol_desired must be positive");
    const int nv = g->shapes[shape_id].nv;
    p.pos.assign(pos, pos + 3 * (size_t)nv);
    p.id = (long long)g->parts.size();
    g->parts.push_back(std::move(p));
    if (pid) *pid = (int)g->parts.size() - 1;
    return BL_OK;
}

int bl_ibm_init(bl_ibm g)
{
    if (!g) return fail(BL_ERR_ARG, "null ibm handle");
    if (g->inited) return fail(BL_ERR_STATE, "bl_ibm_init: already initialised");
    bl_lattice L = g->lat;
    int rc = ensure_force_field(L);
    if (rc) return rc;
    // shapes
    std::vector<int> s_voff{0}, s_toff{0}, s_loff{0}, s_poff{0}, s_vtoff{0}, s_vloff{0}, s_vpoff{0};
    std::vector<int> s_tri, s_link, s_pair, vt_head, vt, vl_head, vl, vp_head, vp;
    std::vector<double> s_area0v, s_geo, s_rest, s_len, s_cs;
    std::vector<double> s_tarea;
    for (const ShapeHost& s : g->shapes) {
        s_voff.push_back(s_voff.back() + s.nv);
        s_toff.push_back(s_toff.back() + s.nt);
        s_loff.push_back(s_loff.back() + s.nl);
        s_poff.push_back(s_poff.back() + s.np);
        s_vtoff.push_back(s_vtoff.back() + (int)s.v_tri.size());
        s_vloff.push_back(s_vloff.back() + (int)s.v_link.size());
        s_vpoff.push_back(s_vpoff.back() + (int)s.v_pair.size());
        s_tri.insert(s_tri.end(), s.tri.begin(), s.tri.end());
        s_tarea.insert(s_tarea.end(), s.tri_area0.begin(), s.tri_area0.end());
        s_geo.insert(s_geo.end(), s.tri_geo0.begin(), s.tri_geo0.end());
        s_rest.insert(s_rest.end(), s.rest.begin(), s.rest.end());
        s_link.insert(s_link.end(), s.link.begin(), s.link.end());
        s_len.insert(s_len.end(), s.link_len.begin(), s.link_len.end());
        s_pair.insert(s_pair.end(), s.pair.begin(), s.pair.end());
        s_cs.insert(s_cs.end(), s.pair_cs0.begin(), s.pair_cs0.end());
        vt_head.insert(vt_head.end(), s.v_tri_off.begin(), s.v_tri_off.end());
        vt.insert(vt.end(), s.v_tri.begin(), s.v_tri.end());
        vl_head.insert(vl_head.end(), s.v_link_off.begin(), s.v_link_off.end());
        vl.insert(vl.end(), s.v_link.begin(), s.v_link.end());
        vp_head.insert(vp_head.end(), s.v_pair_off.begin(), s.v_pair_off.end());
        vp.insert(vp.end(), s.v_pair.begin(), s.v_pair.end());
        s_area0v.push_back(s.area);
    }
    g->nshape = (int)g->shapes.size();
    if ((rc = upload(g->s_voff, s_voff)) || (rc = upload(g->s_toff, s_toff)) || (rc = upload(g->s_loff, s_loff)) ||
        (rc = upload(g->s_poff, s_poff)) || (rc = upload(g->s_vtoff, s_vtoff)) || (rc = upload(g->s_vloff, s_vloff)) ||
        (rc = upload(g->s_vpoff, s_vpoff)) || (rc = upload(g->s_tri, s_tri)) || (rc = upload(g->s_tri_area0, s_tarea)) ||
        (rc = upload(g->s_tri_geo0, s_geo)) || (rc = upload(g->s_rest, s_rest)) || (rc = upload(g->s_link, s_link)) ||
        (rc = upload(g->s_link_len, s_len)) || (rc = upload(g->s_pair, s_pair)) || (rc = upload(g->s_pair_cs0, s_cs)) ||
        (rc = upload(g->s_vt_head, vt_head)) || (rc = upload(g->s_vt, vt)) || (rc = upload(g->s_vl_head, vl_head)) ||
        (rc = upload(g->s_vl, vl)) || (rc = upload(g->s_vp_head, vp_head)) || (rc = upload(g->s_vp, vp)) ||
        (rc = upload(g->s_area0, s_area0v)))
        return rc;
    // particles
    g->np = (int)g->parts.size();
    std::vector<long> voff{0}, toff{0}, loff{0}, poff{0};
    std::vector<int> pshape, pmodel, pbug;
    std::vector<double> params, pos;
    for (const auto& p : g->parts) {
        const ShapeHost& s = g->shapes[p.shape];
        voff.push_back(voff.back() + s.nv);
        toff.push_back(toff.back() + s.nt);
        loff.push_back(loff.back() + s.nl);
        poff.push_back(poff.back() + s.np);
        pshape.push_back(p.shape);
        pmodel.push_back(p.model);
        pbug.push_back(p.bug);
        params.insert(params.end(), p.params, p.params + 8);
        pos.insert(pos.end(), p.pos.begin(), p.pos.end());
    }
    g->NV = voff.back();
    if (g->NV >= (1L << 29)) return fail(BL_ERR_CAPACITY, "bl_ibm_init: at most 2^29 vertices");
    g->NT = toff.back();
    g->NL = loff.back();
    g->NP = poff.back();
    {
        std::vector<int> vp, tp, rp, lp;
        vp.reserve(g->NV);
        tp.reserve(g->NT);
        rp.reserve(g->NP);
        lp.reserve(g->NL);
        for (int p = 0; p < g->np; ++p) {
            vp.insert(vp.end(), voff[p + 1] - voff[p], p);
            tp.insert(tp.end(), toff[p + 1] - toff[p], p);
            rp.insert(rp.end(), poff[p + 1] - poff[p], p);
            lp.insert(lp.end(), loff[p + 1] - loff[p], p);
        }
        // per vertex: where its link / triangle / pair incidence lists start
        // in the concatenated lists and how many entries its particle's
        // model uses (links for RBCs, pairs for RBCs and model 3), and the
        // particle
        std::vector<int> inc;
        inc.reserve(8 * (size_t)g->NV);
        for (int p = 0; p < g->np; ++p) {
            const int sh = g->parts[p].shape, model = g->parts[p].model;
            const ShapeHost& S = g->shapes[sh];
            const bool links = model == BL_MODEL_RBC, pairs = model == BL_MODEL_RBC || model == 3;
            for (int i = 0; i < S.nv; ++i) {
                inc.push_back(s_vloff[sh] + S.v_link_off[i]);
                inc.push_back(links ? S.v_link_off[i + 1] - S.v_link_off[i] : 0);
                inc.push_back(s_vtoff[sh] + S.v_tri_off[i]);
                inc.push_back(S.v_tri_off[i + 1] - S.v_tri_off[i]);
                inc.push_back(s_vpoff[sh] + S.v_pair_off[i]);
                inc.push_back(pairs ? S.v_pair_off[i + 1] - S.v_pair_off[i] : 0);
                inc.push_back(p);
                inc.push_back(0);
            }
        }
        if ((rc = upload(g->v_part, vp)) || (rc = upload(g->t_part, tp)) || (rc = upload(g->r_part, rp)) ||
            (rc = upload(g->l_part, lp)) || (rc = upload(g->v_inc, inc)))
            return rc;
    }
    // vertex reals: FP32 with reduced-precision populations; rigid particles
    // (their own FP64 dynamics, no fluid coupling) keep FP64
    bool any_rigid = false;
    for (const auto& p : g->parts) any_rigid = any_rigid || p.model == BL_MODEL_RIGID;
    g->vreal = (L->storage == BL_STORE_F64 || any_rigid) ? 8 : 4;
    const size_t vr = (size_t)g->vreal;
    const size_t nec = 9 * (size_t)g->NT + 12 * (size_t)g->NP + 3 * (size_t)g->NL;
    if ((rc = upload(g->p_voff, voff)) || (rc = upload(g->p_toff, toff)) || (rc = upload(g->p_loff, loff)) ||
        (rc = upload(g->p_poff, poff)) || (rc = upload(g->p_shape, pshape)) || (rc = upload(g->p_model, pmodel)) ||
        (rc = upload(g->p_bug, pbug)) || (rc = upload(g->p_params, params)) ||
        (rc = alloc_bytes(g->pos, vr * 3 * g->NV)) || (rc = alloc_bytes(g->vel, vr * 3 * g->NV)) ||
        (rc = alloc_bytes(g->force, vr * 3 * g->NV)) || (rc = alloc(g->p_geom, kGeomSums * (size_t)g->np)) ||
        (rc = alloc(g->p_delta, 3 * (size_t)g->np)) || (rc = alloc_bytes(g->ec, vr * nec)) ||
        (rc = alloc_bytes(g->v_pos0, vr * 4 * g->NV)))
        return rc;
    if ((rc = vreal_upload(g, g->pos, 0, pos.data(), (long)pos.size(), L->stream))) return rc;
    g->ec_pair = 9 * g->NT;
    g->ec_link = g->ec_pair + 12 * g->NP;
    // The clears below run on the lattice's stream, as what follows them does:
    // it does not wait for the null stream, and a clear there may still be
    // under way when the call returns.
    {
        const size_t csz = L->storage == BL_STORE_F64 ? sizeof(Vel4<double>) : sizeof(Vel4<float>);
        g->ut = nullptr;
        BL_HIP(hipMalloc(&g->ut, csz * (size_t)L->ncell));
        BL_HIP(hipMemsetAsync(g->ut, 0, csz * (size_t)L->ncell, L->stream));
    }
    BL_HIP(hipMemsetAsync(g->vel, 0, vr * 3 * std::max<long>(g->NV, 1), L->stream));
    BL_HIP(hipMemsetAsync(g->force, 0, vr * 3 * std::max<long>(g->NV, 1), L->stream));
    {  // vertex velocities and forces of particles loaded from a checkpoint
        long v0 = 0;
        for (const auto& p : g->parts) {
            const long n = (long)p.pos.size();
            if ((long)p.vel.size() == n && (rc = vreal_upload(g, g->vel, 3 * v0, p.vel.data(), n, L->stream)))
                return rc;
            if ((long)p.force.size() == n && (rc = vreal_upload(g, g->force, 3 * v0, p.force.data(), n, L->stream)))
                return rc;
            v0 += n / 3;
        }
    }
    // tiles
    if ((rc = alloc(g->tile_count, L->ntiles)) || (rc = alloc(g->tile_list, (size_t)L->ntiles * kTileCap)) ||
        (rc = alloc(g->active, 4 * (size_t)L->ntiles)) || (rc = alloc(g->n_active, 16)))
        return rc;
    BL_HIP(hipMemsetAsync(g->n_active, 0, 16 * sizeof(int), L->stream));
    if ((rc = alloc(g->flags_alt, L->ntiles))) return rc;
    BL_HIP(hipMemsetAsync(g->flags_alt, 0, L->ntiles, L->stream));
    BL_HIP(hipMalloc(&g->force_alt, 3 * L->stride * L->force_bytes));
    BL_HIP(hipMemsetAsync(g->force_alt, 0, 3 * L->stride * L->force_bytes, L->stream));
    {
        // chunks of 256 triangles per particle
        std::vector<int> choff{0}, tab, tvert;
        tvert.reserve(3 * (size_t)g->NT);
        for (int p = 0; p < g->np; ++p) {
            const ShapeHost& S = g->shapes[g->parts[p].shape];
            const long nt = toff[p + 1] - toff[p];
            const int nch = (int)std::max<long>(1, (nt + 255) / 256);
            for (int k = 0; k < nch; ++k) {
                tab.push_back((int)(toff[p] + 256L * k));
                tab.push_back((int)std::max<long>(0, std::min<long>(256, nt - 256L * k)));
            }
            choff.push_back(choff.back() + nch);
            for (long t = 0; t < 3 * nt; ++t) tvert.push_back((int)(voff[p] + S.tri[t]));
        }
        g->nchunk = (int)tab.size() / 2;
        g->geom_one = true;
        for (int p = 0; p < g->np; ++p) g->geom_one = g->geom_one && toff[p + 1] - toff[p] <= kGeomTriangles;
        if ((rc = upload(g->p_choff, choff)) || (rc = upload(g->ch_tab, tab)) || (rc = upload(g->t_vert, tvert)) ||
            (rc = alloc(g->ch_partial, kGeomSums * (size_t)std::max(g->nchunk, 1))))
            return rc;
    }
    BL_HIP(hipMemsetAsync(g->tile_count, 0, L->ntiles * sizeof(int), L->stream));
    // voxelization
    const size_t nbits = (size_t)L->nx * L->ny * column_words(L->nz);
    g->hit_cap = std::max<long>(64 * g->NT, 1024);
    if ((rc = alloc(g->col_bits, nbits)) || (rc = alloc(g->n_hits, 1)) || (rc = alloc(g->phase, L->ncell))) return rc;
    BL_HIP(hipMemsetAsync(g->col_bits, 0, nbits * sizeof(unsigned), L->stream));
    BL_HIP(hipMemsetAsync(g->n_hits, 0, sizeof(int), L->stream));
    BL_HIP(hipMemsetAsync(g->phase, 0, L->ncell, L->stream));
    for (auto& e : g->ev) BL_HIP(hipEventCreate(&e));
    for (auto& st : g->aux) BL_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    for (auto& e : g->fev) BL_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    g->inited = true;
    if ((rc = alloc_near(g))) return rc;
    if (!g->pp.empty() && (rc = interactions_alloc(g))) return rc;
    // update() of every particle and the centre-of-mass mapping of add_particle
    // (rigid particles map their own centre, rigid_init)
    rc = update_particles(g, 1);
    if (rc) return rc;
    if ((rc = rigid_init(g))) return rc;
    BL_HIP(hipStreamSynchronize(L->stream));
    return BL_OK;
}

int bl_ibm_set_boundary(bl_ibm g, const bl_boundary* b)
{
    if (!g) return fail(BL_ERR_ARG, "null ibm handle");
    if (b && b->kind != BL_BOUNDARY_PIPE && b->kind != BL_BOUNDARY_PLATES)
        return fail(BL_ERR_ARG, "bl_ibm_set_boundary: unknown boundary kind");
    if (g->lat) BL_HIP(hipStreamSynchronize(g->lat->stream));
    g->has_boundary = b != nullptr;
    if (b) g->boundary = *b;
    ibm_invalidate_graphs(g);
    return alloc_near(g);
}

int bl_ibm_interpolate(bl_ibm g)
{
    int rc = need_stencil(g);
    return rc ? rc : do_interpolate(g);
}

int bl_ibm_compute_forces(bl_ibm g)
{
    int rc = need_init(g);
    if (!rc) rc = rigid_refuse_coupling(g);
    return rc ? rc : do_forces(g, g->lat->stream);
}

int bl_ibm_spread(bl_ibm g)
{
    int rc = need_stencil(g);
    if (rc) return rc;
    if ((rc = do_spread(g))) return rc;
    return check_overflow(g);
}

int bl_ibm_move(bl_ibm g)
{
    int rc = need_init(g);
    if (!rc) rc = rigid_refuse_coupling(g);
    if (rc) return rc;
    if ((rc = do_move(g))) return rc;
    return do_voxelize(g, g->lat->stream);
}

int bl_ibm_step(bl_ibm g)
{
    int rc = need_stencil(g);
    if (rc) return rc;
    g->timing = true;
    rc = step_serial(g);
    g->timing = false;
    if (rc) return rc;
    BL_HIP(hipEventSynchronize(g->ev[5]));
    for (int k = 0; k < 5; ++k) {
        float ms = 0.f;
        hipEventElapsedTime(&ms, g->ev[k], g->ev[k + 1]);
        g->stage_ms[k] = ms;
    }
    return check_overflow(g);
}

namespace {
constexpr int kLongRun = 32;  // steps per replay of the long captured run

// Captures `n` (even) coupled steps into graph slot `slot` unless the slot
// holds a capture made in the same step parity / buffer / list-reset state
// and the same lattice and boundary generations (no setter ran since).
int ensure_graph(bl_ibm g, int slot, int n)
{
    bl_lattice L = g->lat;
    const long long par = (L->steps & 1) | ((long long)g->alt << 1) | ((long long)g->prepped << 2);
    if (g->graph[slot] && g->graph_parity[slot] == par && g->graph_gen[slot][0] == L->gen &&
        g->graph_gen[slot][1] == g->gen)
        return BL_OK;
    if (g->graph[slot]) {
        hipGraphExecDestroy(g->graph[slot]);
        g->graph[slot] = nullptr;
    }
    hipGraph_t graph;
    BL_HIP(hipStreamBeginCapture(L->stream, hipStreamCaptureModeThreadLocal));
    const long long s0 = L->steps;
    int rc = steps_forked(g, n);
    hipError_t e = hipStreamEndCapture(L->stream, &graph);
    L->steps = s0;  // capture did not execute anything
    if (rc) return rc;
    if (e != hipSuccess) return fail(BL_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    e = hipGraphInstantiate(&g->graph[slot], graph, nullptr, nullptr, 0);
    hipGraphDestroy(graph);
    if (e != hipSuccess) return fail(BL_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
    g->graph_parity[slot] = par;
    // after the capture: a capture that set state for the first time (the
    // phase field of a voxelization) keys on the state it captured
    g->graph_gen[slot][0] = L->gen;
    g->graph_gen[slot][1] = g->gen;
    return BL_OK;
}

int replay(bl_ibm g, int slot, int n, int reps)
{
    for (int r = 0; r < reps; ++r) {
        BL_HIP(hipGraphLaunch(g->graph[slot], g->lat->stream));
        g->lat->steps += n;
    }
    return BL_OK;
}
}  // namespace

int bl_coupled_steps(bl_ibm g, int n_steps, int use_graph)
{
    int rc = need_stencil(g);
    if (rc) return rc;
    bl_lattice L = g->lat;
    if (n_steps < 0) return fail(BL_ERR_ARG, "bl_coupled_steps: negative step count");
    int done = 0;
    // a force field loaded into the lattice is consumed over the next two
    // steps; those run eagerly, so no captured step depends on it
    for (; done < n_steps && ibm_needs_settle(g); ++done)
        if ((rc = steps_forked(g, 1))) return rc;
    if (use_graph) {
        // Runs of kLongRun steps, then pairs (the two AA parities), each
        // captured once per step parity and replayed.
        const int left = n_steps - done;
        if (left >= kLongRun) {
            if ((rc = ensure_graph(g, 1, kLongRun))) return rc;
            if ((rc = replay(g, 1, kLongRun, left / kLongRun))) return rc;
            done += left / kLongRun * kLongRun;
        }
        if (n_steps - done >= 2) {
            if ((rc = ensure_graph(g, 0, 2))) return rc;
            const int reps = (n_steps - done) / 2;
            if ((rc = replay(g, 0, 2, reps))) return rc;
            done += 2 * reps;
        }
    }
    if (done < n_steps && (rc = steps_forked(g, n_steps - done))) return rc;
    return check_overflow(g);
}

int bl_coupled_prepare(bl_ibm g, int n_steps)
{
    int rc = need_stencil(g);
    if (rc) return rc;
    if (n_steps < 0) return fail(BL_ERR_ARG, "bl_coupled_prepare: negative step count");
    if (ibm_needs_settle(g))
        return fail(BL_ERR_STATE, "bl_coupled_prepare: the next step runs eagerly (a loaded force field or a changed "
                                  "body force); run it first");
    // the graphs bl_coupled_steps(g, n_steps, 1) replays from this state: runs
    // of kLongRun steps keep the step parity, so both are captured for it
    if (n_steps >= kLongRun && (rc = ensure_graph(g, 1, kLongRun))) return rc;
    if (n_steps % kLongRun >= 2 && (rc = ensure_graph(g, 0, 2))) return rc;
    return BL_OK;
}

int bl_ibm_count(bl_ibm g, int* particles, int* vertices)
{
    if (!g) return fail(BL_ERR_ARG, "null ibm handle");
    if (particles) *particles = (int)g->parts.size();
    long nv = 0;
    for (const auto& p : g->parts) nv += g->shapes[p.shape].nv;
    if (vertices) *vertices = (int)nv;
    return BL_OK;
}

int bl_particle_get(bl_ibm g, int pid, int what, double* out)
{
    int rc = need_init(g);
    if (rc) return rc;
    if (!out || what < 0 || what > 2 || pid < -1 || pid >= g->np) return fail(BL_ERR_ARG, "bl_particle_get: bad argument");
    std::vector<long> voff{0};
    for (const auto& p : g->parts) voff.push_back(voff.back() + g->shapes[p.shape].nv);
    const long v0 = pid < 0 ? 0 : voff[pid], v1 = pid < 0 ? voff.back() : voff[pid + 1];
    const void* src = what == 0 ? g->pos : (what == 1 ? g->vel : g->force);
    return vreal_download(g, out, src, 3 * v0, 3 * (v1 - v0), g->lat->stream);
}

int bl_particle_set_positions(bl_ibm g, int pid, const double* pos)
{
    int rc = need_init(g);
    if (rc) return rc;
    if (!pos || pid < -1 || pid >= g->np) return fail(BL_ERR_ARG, "bl_particle_set_positions: bad argument");
    std::vector<long> voff{0};
    for (const auto& p : g->parts) voff.push_back(voff.back() + g->shapes[p.shape].nv);
    const long v0 = pid < 0 ? 0 : voff[pid], v1 = pid < 0 ? voff.back() : voff[pid + 1];
    if ((rc = vreal_upload(g, g->pos, 3 * v0, pos, 3 * (v1 - v0), g->lat->stream))) return rc;
    rc = update_particles(g, 0);
    if (rc) return rc;
    BL_HIP(hipStreamSynchronize(g->lat->stream));
    return BL_OK;
}

}  // extern "C"

namespace {
// Membrane forces alone (RBCParticle::compute_forces): no decorators, no
// particle-particle forces.
int membrane_forces(bl_ibm g, hipStream_t s)
{
    launch_membrane(g, s, false);
    BL_CHECK_LAUNCH();
    return BL_OK;
}

// One calibration step (node masses, then the relax update) of the
// selected particles.
int calib_step(bl_ibm g, hipStream_t s, const int* active, const double* damp, const double* v0, const double* v1,
               int n_it, double* mass, int* step)
{
    with_vreal(g, [&](auto tag) {
        using R = decltype(tag);
        hipLaunchKernelGGL(k_calib_mass<R>, dim3(nblk(g->NV)), dim3(256), 0, s, force_view<R>(g), g->NV, active, mass,
                           step);
        hipLaunchKernelGGL(k_calib_relax<R>, dim3(nblk(g->NV)), dim3(256), 0, s, g->NV, (const int*)g->v_part,
                           (const long*)g->p_voff, active, damp, v0, v1, n_it, (const int*)step, (const double*)mass,
                           (const R*)g->force, (R*)g->vel, (R*)g->pos, g->p_params);
        return 0;
    });
    BL_CHECK_LAUNCH();
    return BL_OK;
}

template <class T>
struct DevBuf {
    T* p = nullptr;
    ~DevBuf() { hipFree(p); }
    int alloc(size_t n)
    {
        BL_HIP(hipMalloc(&p, sizeof(T) * std::max<size_t>(n, 1)));
        return BL_OK;
    }
};
}  // namespace

extern "C" {

int bl_rbc_shrink_volume(bl_ibm g, int pid, double vol_final, int n_it, double damping, double* damping_out)
{
    int rc = need_init(g);
    if (rc) return rc;
    if (pid < -1 || pid >= g->np) return fail(BL_ERR_ARG, "bl_rbc_shrink_volume: bad particle id");
    if (n_it < 1 || !(damping > 0) || !(vol_final > 0))
        return fail(BL_ERR_ARG, "bl_rbc_shrink_volume: need n_it >= 1, damping > 0, vol_final > 0");
    const int np = g->np;
    std::vector<int> todo(np, 0);
    std::vector<double> damp(np, damping), v0(np, 0.0), v1(np, vol_final);
    std::vector<long> voff(np + 1, 0);
    for (int p = 0; p < np; ++p) {
        const auto& P = g->parts[p];
        voff[p + 1] = voff[p] + g->shapes[P.shape].nv;
        v0[p] = g->shapes[P.shape].volume;  // the rest shape's volume
        const bool rbc = P.model == BL_MODEL_RBC || P.model == 3;
        if (pid == p && !rbc) return fail(BL_ERR_ARG, "bl_rbc_shrink_volume: the particle has no volume constraint");
        todo[p] = (pid == -1 || pid == p) && rbc;
    }
    hipStream_t s = g->lat->stream;
    const size_t nv3 = 3 * (size_t)g->NV;
    const size_t vr = (size_t)g->vreal;
    DevBuf<int> d_active, d_step;
    DevBuf<double> d_damp, d_v0, d_v1, d_mass, prm0;
    DevBuf<char> pos0, vel0, frc0;  // the vertex state, in the boundary's reals
    if ((rc = d_active.alloc(np)) || (rc = d_step.alloc(1)) || (rc = d_damp.alloc(np)) || (rc = d_v0.alloc(np)) ||
        (rc = d_v1.alloc(np)) || (rc = d_mass.alloc(g->NV)) || (rc = pos0.alloc(vr * nv3)) ||
        (rc = vel0.alloc(vr * nv3)) || (rc = frc0.alloc(vr * nv3)) || (rc = prm0.alloc(8 * (size_t)np)))
        return rc;
    BL_HIP(hipMemcpyAsync(d_v0.p, v0.data(), sizeof(double) * np, hipMemcpyHostToDevice, s));
    BL_HIP(hipMemcpyAsync(d_v1.p, v1.data(), sizeof(double) * np, hipMemcpyHostToDevice, s));
    // the starting state: geometry and forces of the current positions with
    // the current parameters (rbc.compute_forces() before the loop)
    if ((rc = update_particles(g, 0, s)) || (rc = membrane_forces(g, s))) return rc;
    BL_HIP(hipMemcpyAsync(pos0.p, g->pos, vr * nv3, hipMemcpyDeviceToDevice, s));
    BL_HIP(hipMemcpyAsync(vel0.p, g->vel, vr * nv3, hipMemcpyDeviceToDevice, s));
    BL_HIP(hipMemcpyAsync(frc0.p, g->force, vr * nv3, hipMemcpyDeviceToDevice, s));
    BL_HIP(hipMemcpyAsync(prm0.p, g->p_params, sizeof(double) * 8 * np, hipMemcpyDeviceToDevice, s));
    for (;;) {
        bool any = false;
        for (int p = 0; p < np; ++p) any = any || todo[p];
        if (!any) break;
        BL_HIP(hipMemcpyAsync(d_active.p, todo.data(), sizeof(int) * np, hipMemcpyHostToDevice, s));
        BL_HIP(hipMemcpyAsync(d_damp.p, damp.data(), sizeof(double) * np, hipMemcpyHostToDevice, s));
        BL_HIP(hipMemsetAsync(d_step.p, 0, sizeof(int), s));
        for (int it = 0; it <= 2 * n_it; ++it) {
            if ((rc = calib_step(g, s, d_active.p, d_damp.p, d_v0.p, d_v1.p, n_it, d_mass.p, d_step.p))) return rc;
            if ((rc = update_particles(g, 0, s)) || (rc = membrane_forces(g, s))) return rc;
        }
        // a particle whose area went NaN starts over with twice the damping
        std::vector<double> geom(kGeomSums * (size_t)np);
        BL_HIP(hipMemcpyAsync(geom.data(), g->p_geom, sizeof(double) * geom.size(), hipMemcpyDeviceToHost, s));
        BL_HIP(hipStreamSynchronize(s));
        for (int p = 0; p < np; ++p) {
            if (!todo[p]) continue;
            const double area = geom[kGeomSums * p];
            if (area == area) {
                todo[p] = 0;
                continue;
            }
            damp[p] *= 2.0;
            const size_t a = vr * 3 * (size_t)voff[p], n = vr * 3 * (size_t)(voff[p + 1] - voff[p]);
            BL_HIP(hipMemcpyAsync((char*)g->pos + a, pos0.p + a, n, hipMemcpyDeviceToDevice, s));
            BL_HIP(hipMemcpyAsync((char*)g->vel + a, vel0.p + a, n, hipMemcpyDeviceToDevice, s));
            BL_HIP(hipMemcpyAsync((char*)g->force + a, frc0.p + a, n, hipMemcpyDeviceToDevice, s));
            BL_HIP(hipMemcpyAsync(g->p_params + 8 * p, prm0.p + 8 * p, sizeof(double) * 8, hipMemcpyDeviceToDevice, s));
            if (damp[p] > 2.0) {  // left in its starting state
                if ((rc = update_particles(g, 0, s))) return rc;
                BL_HIP(hipStreamSynchronize(s));
                return fail(BL_ERR_STATE, "bl_rbc_shrink_volume: particle " + std::to_string(p) +
                                              " diverges for every damping up to 2");
            }
        }
        // restored particles need their geometry back before the next attempt
        if ((rc = update_particles(g, 0, s))) return rc;
    }
    // the calibrated vol_desired stays with the particles (host copy too)
    std::vector<double> prm(8 * (size_t)np);
    BL_HIP(hipMemcpyAsync(prm.data(), g->p_params, sizeof(double) * prm.size(), hipMemcpyDeviceToHost, s));
    BL_HIP(hipStreamSynchronize(s));
    for (int p = 0; p < np; ++p) {
        for (int k = 0; k < 8; ++k) g->parts[p].params[k] = prm[8 * p + k];
        if (damping_out) damping_out[p] = damp[p];
    }
    g->binned = false;
    ibm_invalidate_graphs(g);
    return BL_OK;
}

int bl_particle_set_state(bl_ibm g, int pid, int what, const double* data)
{
    int rc = need_init(g);
    if (rc) return rc;
    if (!data || what < 0 || what > 2 || pid < -1 || pid >= g->np)
        return fail(BL_ERR_ARG, "bl_particle_set_state: bad argument");
    if (what == 0) return bl_particle_set_positions(g, pid, data);
    long v0 = 0, v1 = 0;
    for (int p = 0; p < g->np; ++p) {
        const long n = g->shapes[g->parts[p].shape].nv;
        if (p < pid) v0 += n;
        if (pid < 0 || p <= pid) v1 += n;
    }
    if (pid < 0) v0 = 0;
    void* dst = what == 1 ? g->vel : g->force;
    return vreal_upload(g, dst, 3 * v0, data, 3 * (v1 - v0), g->lat->stream);
}

int bl_particle_set_params(bl_ibm g, int pid, const double* params, int nparams)
{
    int rc = need_init(g);
    if (rc) return rc;
    if (!params || pid < 0 || pid >= g->np || nparams < 1 || nparams > 8)
        return fail(BL_ERR_ARG, "bl_particle_set_params: bad argument");
    double* h = g->parts[pid].params;
    for (int k = 0; k < nparams; ++k) h[k] = params[k];
    BL_HIP(hipMemcpyAsync(g->p_params + 8 * (size_t)pid, h, sizeof(double) * 8, hipMemcpyHostToDevice, g->lat->stream));
    BL_HIP(hipStreamSynchronize(g->lat->stream));
    ibm_invalidate_graphs(g);
    return BL_OK;
}

int bl_rbc_relax_nodes(bl_ibm g, int pid, double damping)
{
    int rc = need_init(g);
    if (rc) return rc;
    if (pid < 0 || pid >= g->np || !(damping >= 0)) return fail(BL_ERR_ARG, "bl_rbc_relax_nodes: bad argument");
    const int model = g->parts[pid].model;
    if (model != BL_MODEL_RBC && model != 3) return fail(BL_ERR_ARG, "bl_rbc_relax_nodes: not a red-cell model");
    hipStream_t s = g->lat->stream;
    const int np = g->np;
    std::vector<int> act(np, 0);
    act[pid] = 1;
    std::vector<double> damp(np, damping);
    DevBuf<int> d_active, d_step;
    DevBuf<double> d_damp, d_mass, d_v;
    if ((rc = d_active.alloc(np)) || (rc = d_step.alloc(1)) || (rc = d_damp.alloc(np)) || (rc = d_mass.alloc(g->NV)) ||
        (rc = d_v.alloc(np)))
        return rc;
    BL_HIP(hipMemcpyAsync(d_active.p, act.data(), sizeof(int) * np, hipMemcpyHostToDevice, s));
    BL_HIP(hipMemcpyAsync(d_damp.p, damp.data(), sizeof(double) * np, hipMemcpyHostToDevice, s));
    BL_HIP(hipMemsetAsync(d_step.p, 0, sizeof(int), s));
    // the vertex forces in place are those of the current positions
    // (compute_forces before the first step); n_it = -1: vol_desired stays
    // as the parameters hold it
    if ((rc = calib_step(g, s, d_active.p, d_damp.p, d_v.p, d_v.p, -1, d_mass.p, d_step.p))) return rc;
    if ((rc = update_particles(g, 0, s)) || (rc = membrane_forces(g, s))) return rc;
    BL_HIP(hipStreamSynchronize(s));
    g->binned = false;
    return BL_OK;
}

int bl_ibm_set_vertex_forces(bl_ibm g, const double* force)
{
    int rc = need_init(g);
    if (rc) return rc;
    hipStream_t s = g->lat->stream;
    if (!force) {
        if (g->has_ext) ibm_invalidate_graphs(g);
        g->has_ext = false;
        return BL_OK;
    }
    if (!g->ext_force) BL_HIP(hipMalloc(&g->ext_force, (size_t)g->vreal * 3 * std::max<long>(g->NV, 1)));
    if ((rc = vreal_upload(g, g->ext_force, 0, force, 3 * g->NV, s))) return rc;
    if (!g->has_ext) ibm_invalidate_graphs(g);
    g->has_ext = true;
    return BL_OK;
}

int bl_particle_membrane_forces(bl_ibm g)
{
    int rc = need_init(g);
    if (rc) return rc;
    hipStream_t s = g->lat->stream;
    if ((rc = update_particles(g, 0, s)) || (rc = membrane_forces(g, s))) return rc;
    BL_HIP(hipStreamSynchronize(s));
    return BL_OK;
}

int bl_particle_observables(bl_ibm g, int pid, double out[14])
{
    int rc = need_init(g);
    if (rc) return rc;
    if (!out || pid < 0 || pid >= g->np) return fail(BL_ERR_ARG, "bl_particle_observables: bad argument");
    double geom[kGeomSums];
    BL_HIP(hipMemcpyAsync(geom, g->p_geom + kGeomSums * pid, sizeof(geom), hipMemcpyDeviceToHost, g->lat->stream));
    const int nv = g->shapes[g->parts[pid].shape].nv;
    std::vector<double> pos(3 * (size_t)nv);
    rc = bl_particle_get(g, pid, 0, pos.data());
    if (rc) return rc;
    // Moment of inertia of the enclosed volume about its centroid
    // (src/fsi/DeformableParticle3D.hh:173-272), FP64 on the host.
    const ShapeHost& s = g->shapes[g->parts[pid].shape];
    double in[10] = {0};
    for (int t = 0; t < s.nt; ++t) {
        const double* v[3] = {&pos[3 * s.tri[3 * t]], &pos[3 * s.tri[3 * t + 1]], &pos[3 * s.tri[3 * t + 2]]};
        const double a[3] = {v[1][0] - v[0][0], v[1][1] - v[0][1], v[1][2] - v[0][2]};
        const double b[3] = {v[2][0] - v[0][0], v[2][1] - v[0][1], v[2][2] - v[0][2]};
        const double N[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]};
        double f1[3], f2[3], f3[3], g0[3], g1[3], g2[3];
        for (int d = 0; d < 3; ++d) {
            const double tmp0 = v[0][d] + v[1][d];
            f1[d] = tmp0 + v[2][d];
            const double tmp1 = v[0][d] * v[0][d];
            const double tmp2 = tmp1 + v[1][d] * tmp0;
            f2[d] = tmp2 + v[2][d] * f1[d];
            f3[d] = v[0][d] * tmp1 + v[1][d] * tmp2 + v[2][d] * f2[d];
            g0[d] = f2[d] + v[0][d] * (f1[d] + v[0][d]);
            g1[d] = f2[d] + v[1][d] * (f1[d] + v[1][d]);
            g2[d] = f2[d] + v[2][d] * (f1[d] + v[2][d]);
        }
        in[0] += N[0] * f1[0];
        in[1] += N[0] * f2[0];
        in[2] += N[1] * f2[1];
        in[3] += N[2] * f2[2];
        in[4] += N[0] * f3[0];
        in[5] += N[1] * f3[1];
        in[6] += N[2] * f3[2];
        in[7] += N[0] * (v[0][1] * g0[0] + v[1][1] * g1[0] + v[2][1] * g2[0]);
        in[8] += N[1] * (v[0][2] * g0[1] + v[1][2] * g1[1] + v[2][2] * g2[1]);
        in[9] += N[2] * (v[0][0] * g0[2] + v[1][0] * g1[2] + v[2][0] * g2[2]);
    }
    in[0] *= 1.0 / 6.0;
    for (int k = 1; k <= 3; ++k) in[k] *= 1.0 / 24.0;
    for (int k = 4; k <= 6; ++k) in[k] *= 1.0 / 60.0;
    for (int k = 7; k <= 9; ++k) in[k] *= 1.0 / 120.0;
    const double V = in[0];
    const double c[3] = {in[1] / V, in[2] / V, in[3] / V};
    double* I = out + 5;
    I[0] = in[5] + in[6] - V * (c[1] * c[1] + c[2] * c[2]);
    I[1] = -in[7] + V * c[0] * c[1];
    I[2] = -in[9] + V * c[2] * c[0];
    I[3] = I[1];
    I[4] = in[4] + in[6] - V * (c[2] * c[2] + c[0] * c[0]);
    I[5] = -in[8] + V * c[1] * c[2];
    I[6] = I[2];
    I[7] = I[5];
    I[8] = in[4] + in[5] - V * (c[0] * c[0] + c[1] * c[1]);
    for (int k = 0; k < 5; ++k) out[k] = geom[k];
    return BL_OK;
}

int bl_ibm_get_phase(bl_ibm g, unsigned char* phase)
{
    int rc = need_init(g);
    if (rc) return rc;
    if (!phase) return fail(BL_ERR_ARG, "bl_ibm_get_phase: null argument");
    BL_HIP(hipMemcpyAsync(phase, g->phase, g->lat->ncell, hipMemcpyDeviceToHost, g->lat->stream));
    BL_HIP(hipStreamSynchronize(g->lat->stream));
    return BL_OK;
}

int bl_ibm_tile_stats(bl_ibm g, long long out[2])
{
    int rc = need_init(g);
    if (rc) return rc;
    if (!out) return fail(BL_ERR_ARG, "bl_ibm_tile_stats: null argument");
    int st[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    BL_HIP(hipMemcpyAsync(st, g->n_active, sizeof(st), hipMemcpyDeviceToHost, g->lat->stream));
    BL_HIP(hipStreamSynchronize(g->lat->stream));
    out[0] = st[g->last_list];
    out[1] = st[5 + g->last_list];
    return BL_OK;
}

int bl_ibm_set_fused_staging(bl_ibm g, int mode)
{
    if (!g) return fail(BL_ERR_ARG, "null ibm handle");
    if (mode < -1 || mode > 1) return fail(BL_ERR_ARG, "bl_ibm_set_fused_staging: mode must be -1, 0 or 1");
    if (mode != g->fused_staging) ibm_invalidate_graphs(g);
    g->fused_staging = mode;
    return BL_OK;
}

int bl_ibm_set_layered(bl_ibm g, int mode)
{
    if (!g) return fail(BL_ERR_ARG, "bl_ibm_set_layered: null handle");
    if (mode < -1 || mode > 1) return fail(BL_ERR_ARG, "bl_ibm_set_layered: mode must be -1, 0 or 1");
    if (mode != g->layered) ibm_invalidate_graphs(g);
    g->layered = mode;
    return BL_OK;
}

int bl_ibm_set_launch(bl_ibm g, const int params[BL_IBM_NLAUNCH])
{
    if (!g || !params) return fail(BL_ERR_ARG, "bl_ibm_set_launch: null argument");
    auto in = [](int v, std::initializer_list<int> ok) { return std::find(ok.begin(), ok.end(), v) != ok.end(); };
    const int* p = params;
    if (!in(p[BL_IBM_BIN_BLOCK], {64, 128, 256}) || !in(p[BL_IBM_ELEM_BLOCK], {64, 128, 256}) ||
        !in(p[BL_IBM_GATHER_LANES], {2, 4, 8}) || !in(p[BL_IBM_INTERP_BLOCK], {64, 128, 256}) ||
        !in(p[BL_IBM_SPREAD_SMALL], {1, 2, 4, 8}) || !in(p[BL_IBM_SPREAD_BIG], {16, 32, 64, 128}) ||
        !in(p[BL_IBM_XCD], {0, 2, 4, 6}))
        return fail(BL_ERR_ARG, "bl_ibm_set_launch: a launch parameter is outside its allowed values");
    bool same = true;
    for (int k = 0; k < BL_IBM_NLAUNCH; ++k) same = same && g->lp[k] == p[k];
    if (same) return BL_OK;
    if (g->lat) BL_HIP(hipStreamSynchronize(g->lat->stream));
    for (int k = 0; k < BL_IBM_NLAUNCH; ++k) g->lp[k] = p[k];
    ibm_invalidate_graphs(g);
    return BL_OK;
}

int bl_ibm_get_launch(bl_ibm g, int params[BL_IBM_NLAUNCH])
{
    if (!g || !params) return fail(BL_ERR_ARG, "bl_ibm_get_launch: null argument");
    for (int k = 0; k < BL_IBM_NLAUNCH; ++k) params[k] = g->lp[k];
    return BL_OK;
}

int bl_ibm_stage_times(bl_ibm g, double out[5])
{
    if (!g || !out) return fail(BL_ERR_ARG, "bl_ibm_stage_times: null argument");
    for (int k = 0; k < 5; ++k) out[k] = g->stage_ms[k];
    return BL_OK;
}

}  // extern "C"
