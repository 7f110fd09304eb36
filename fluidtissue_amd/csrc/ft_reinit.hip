// ft_reinit.hip -- gfx950 level-set reinitialization behind the C ABI of
// include/ftreinit.h.
//
// Pipeline of one reinit (LevelSet::resetPhi_, src/fem/LevelSet.cpp:429-455),
// all on the device, mesh resident in HBM:
//   1 k_node_signs    phi -> sign bitmap (1 bit/node)
//   2 k_classify      one pass over all tets: crossing bitmap + per-block
//                     (crossing tets, triangles) counts      (LevelSet.cpp:377-383)
//   3 scan            block counts -> exclusive offsets
//   4 k_compact       crossing tets in increasing tet order + triangle offsets
//   5 k_xtet          crossing tets: t2e/edges -> crossing edges in t2e order,
//                     checked, marked in an edge bitmap       (LevelSet.cpp:385-405)
//   6 scan            edge-bitmap popcounts -> rank of each crossing edge, i.e.
//                     the ifp index in increasing edge order  (LevelSet.cpp:278-299)
//   7 k_points        FP64 crossing points, ifp2e, retained-node bitmap
//                                                            (LevelSet.cpp:281-298, 443-447)
//   8 k_tris          triangles in tet order with the reference's orientation
//                     rule, normal lengths                   (LevelSet.cpp:330-347, 393-399)
//   9 p2t / area      per-point triangle lists (CSR, ascending) and the
//                     ordered area sums                      (LevelSet.cpp:349-356)
//  10 index           primitives (points or triangles) sorted by uniform bin,
//                     leaves = non-empty bins in Morton order, 64-ary tree of
//                     oriented boxes over the leaves
//  11 schedule        64-node tiles deep inside the surface listed first
//                     (k_tile_deep, scan, k_tile_list; full domain only)
//  12 k_query         per node (Morton-sorted order): exact nearest primitive
//                     (triangles: FP32 search, FP64 settle of the best two),
//                     sign from phi < 0, retained values and the blend fused
//                     in the epilogue (EuclideanDistance.cu:45-58,
//                     LevelSet.cpp:438-448, 74, 148)
// The whole file is compiled with -ffp-contract=off: products and sums are
// rounded one at a time unless an fma is written out, so the bit-exact parts
// (interpolation, orientation, areas, point distances) match the oracle.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <type_traits>
#include <vector>

#include "ftreinit.h"
#include "ft_device.hpp"
#include "ft_internal.hpp"
#include "ft_p2t.hpp"

using ftd::Grid;
using ftd::TriRec;

namespace {

constexpr int kBS = 256;                 // threads per block of the streaming kernels
constexpr int kScanTile = 2048;          // elements per scan block (256 x 8)
constexpr int kMaxBinsLog2PerAxis = 8;   // <= 256 bins per axis, 2^24 Morton cells

#define FT_HIP(call)                                                                   \
    do {                                                                               \
        hipError_t e_ = (call);                                                        \
        if (e_ != hipSuccess)                                                          \
            return ft::set_error(FT_ERR_HIP, "%s failed: %s", #call, hipGetErrorString(e_)); \
    } while (0)

#define FT_TRY(...)                     \
    do {                                \
        int rc_ = (__VA_ARGS__);        \
        if (rc_ != FT_OK) return rc_;   \
    } while (0)

inline unsigned grid1d(int64_t n, int bs = kBS) { return (unsigned)((n + bs - 1) / bs); }

// Scalar slots of a handle (a small device u64 array): stage totals written
// by the scans, the error word, capacity and traversal overflow flags.
//   S_BLK    (crossing tets << 32) | triangles
//   S_EDGES  crossing points (low 32 bits)
//   S_ERR    ~0, or (code << 40) | first failing tet
//   S_BINS   leaves of the index (low 32 bits)
//   S_DEEP   query tiles scheduled first (low 32 bits), of which the very deep
//            ones, split over several waves (high 32 bits); in a narrow band
//            the tiles to search (k_tile_near)
//   S_CAP    a stage total exceeded the capacity its buffers were sized for
//   S_LV     3 slots: primitives and tree nodes per level (ftd::Lv)
//   S_CLAMP  nodes clamped to the band, of a single field
// (S_TOP of them are read back), and after them
//   S_Q      the query's counters (9 x u32: deep tiles, then one per XCD),
//            zeroed per launch, each in a line of its own: in one line their
//            atomics wait for each other (crossing points at 256^3 3.55 ms against
//            3.15, a 256^3 band 3.59 against 1.90)
enum Slot { S_BLK = 0, S_EDGES = 1, S_ERR = 2, S_P2T = 3, S_BINS = 4, S_DEEP = 5, S_CAP = 6,
            S_LV = 7, S_CLAMP = 10, S_TOP = 16, S_Q = S_TOP, S_N = S_Q + 9 * 16 };
constexpr int kQueueLine = 32;           // words between the query's counters

// Stage totals of the running reinit as the kernels see them.  Kernels after
// a scan read the total from the device, so a launch sized for a capacity
// (a replayed graph) processes exactly this call's elements.
__device__ __forceinline__ int64_t cnt_xtets(const uint64_t* sc) { return (int64_t)(sc[S_BLK] >> 32); }
__device__ __forceinline__ int64_t cnt_tris(const uint64_t* sc) { return (int64_t)(sc[S_BLK] & 0xffffffffull); }
__device__ __forceinline__ int64_t cnt_points(const uint64_t* sc) { return (int64_t)(sc[S_EDGES] & 0xffffffffull); }
__device__ __forceinline__ int64_t cnt_leaves(const uint64_t* sc) { return (int64_t)(sc[S_BINS] & 0xffffffffull); }
// Set once a stage failed (t2e or degenerate tet) or outgrew its buffers:
// every later kernel of the reinit then does nothing and phi stays as it was.
__device__ __forceinline__ bool halted(const uint64_t* sc)
{
    return sc[S_CAP] != 0ull || sc[S_ERR] != ~0ull;
}

// Connectivity of the resident fields as the marching-tets kernels see it:
// one concatenated array per kind (global indices), or, for a batch of
// resident meshes, each field's own arrays read in place (field-local
// indices, to which the field's node or edge offset is added), so that a
// batch is assembled without copying its tets, t2e and edges.
struct MeshView {
    const int4* tets;                // concatenated (null: per field)
    const int2* t2e3;                // t2e rows as 3 int2
    const int2* edges;
    const int4* const* f_tets;       // per field
    const int2* const* f_t2e3;
    const int2* const* f_edges;
    const int64_t* node_off;         // device offsets, nf + 1 each
    const int64_t* tet_off;
    const int64_t* edge_off;
    int nf;
};

// Field of tet t (t < T) and of edge e: binary search over the offsets.
__device__ __forceinline__ int mv_tet_field(const MeshView& m, int64_t t)
{
    return ftd::field_of(m.tet_off, m.nf, t);
}
__device__ __forceinline__ int mv_edge_field(const MeshView& m, int64_t e)
{
    return ftd::field_of(m.edge_off, m.nf, e);
}
// Tet t of field k (k = its field) with global node ids.
__device__ __forceinline__ int4 mv_tet(const MeshView& m, int64_t t, int k)
{
    if (m.tets) return m.tets[t];
    int4 q = m.f_tets[k][t - m.tet_off[k]];
    const int32_t a = (int32_t)m.node_off[k];
    q.x += a; q.y += a; q.z += a; q.w += a;
    return q;
}
// Row j (0..2) of tet t's t2e, as two global edge ids.
__device__ __forceinline__ int2 mv_t2e(const MeshView& m, int64_t t, int j, int k)
{
    if (m.t2e3) return m.t2e3[3 * t + j];
    int2 r = m.f_t2e3[k][3 * (t - m.tet_off[k]) + j];
    const int32_t a = (int32_t)m.edge_off[k];
    r.x += a; r.y += a;
    return r;
}
// Edge e of field k with global node ids.
__device__ __forceinline__ int2 mv_edge(const MeshView& m, int64_t e, int k)
{
    if (m.edges) return m.edges[e];
    int2 ab = m.f_edges[k][e - m.edge_off[k]];
    const int32_t a = (int32_t)m.node_off[k];
    ab.x += a; ab.y += a;
    return ab;
}

// ============================================================================
// Generic kernels: fill and exclusive scan
// ============================================================================
template <class T>
__global__ __launch_bounds__(kBS) void k_fill(T* p, int64_t n, T v)
{
    const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (i < n) p[i] = v;
}

// Several ranges of 4-byte words set in one launch (what a stage needs cleared).
struct WordRanges {
    static constexpr int kMax = 8;
    uint32_t* p[kMax];
    int64_t end[kMax];               // words of the ranges up to and including this one
    uint32_t v[kMax];
    int n = 0;
    void add(void* at, int64_t words, uint32_t value)
    {
        if (words <= 0) return;
        p[n] = static_cast<uint32_t*>(at);
        end[n] = total() + words;
        v[n++] = value;
    }
    int64_t total() const { return n ? end[n - 1] : 0; }
};
__global__ __launch_bounds__(kBS) void k_set_words(WordRanges r)
{
    const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
    int64_t lo = 0;
    for (int k = 0; k < r.n; k++) {
        if (i < r.end[k]) {
            r.p[k][i - lo] = r.v[k];
            return;
        }
        lo = r.end[k];
    }
}

// clear: the scan leaves zeros in its input (cursors of the pass that follows).
struct LoadSame {
    static constexpr bool clear = false;
    template <class T> __device__ T operator()(T v) const { return v; }
};
struct LoadClear : LoadSame {
    static constexpr bool clear = true;
};
struct LoadPopc {  // u64 bitmap word -> popcount
    static constexpr bool clear = false;
    __device__ uint32_t operator()(uint64_t v) const { return (uint32_t)__popcll(v); }
};
// A scan of a field's nodes per bin that also gives the query tiles (64 slots)
// of each block of cpb consecutive bins, from the sums of the threads' runs
// (setting up a batch of 24 grids of 26^3 to 96^3 takes 2.22 ms, with a pass of
// its own over the offsets 2.35).
struct LoadBlocks : LoadSame {
    int cpb;                         // a multiple of a run, at most 64 lanes' worth
    uint32_t* tiles;
    LoadBlocks(int c, uint32_t* t) : cpb(c), tiles(t) {}
    template <int RUN>
    __device__ __forceinline__ void sums(int64_t base, int64_t n, uint32_t s) const
    {
        const int lanes = cpb / RUN;
        for (int o = 1; o < lanes; o <<= 1) s += __shfl_xor(s, o);
        if (base < n && base % cpb == 0) tiles[base / cpb] = (s + 63u) / 64u;
    }
};
struct LoadTileClass {  // tile class 0 / 1 deep / 2 very deep -> (very deep << 32) | deep
    static constexpr bool clear = false;
    __device__ uint64_t operator()(uint32_t c) const { return ((uint64_t)(c == 2) << 32) | (uint64_t)(c >= 1); }
};

template <class TI, class TO, class Ld>
__global__ __launch_bounds__(kBS) void k_scan_reduce(const TI* in, int64_t n, TO* bsum, Ld ld)
{
    __shared__ TO lds[kBS / 64 + 1];
    const int64_t base = (int64_t)blockIdx.x * kScanTile;
    TO s = 0;
#pragma unroll
    for (int k = 0; k < kScanTile / kBS; k++) {
        const int64_t i = base + (int64_t)k * kBS + threadIdx.x;
        if (i < n) s += (TO)ld(in[i]);
    }
    TO tot;
    ftd::block_excl_scan<TO, kBS>(s, lds, &tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

template <class TO>
__global__ __launch_bounds__(1024) void k_scan_top(TO* bsum, int64_t nb, TO* total)
{
    __shared__ TO lds[1024 / 64 + 1];
    TO carry = TO(0);
    for (int64_t c = 0; c < nb; c += 1024) {
        const int64_t i = c + threadIdx.x;
        const TO v = i < nb ? bsum[i] : TO(0);
        TO tot;
        const TO ex = ftd::block_excl_scan<TO, 1024>(v, lds, &tot);
        if (i < nb) bsum[i] = ex + carry;
        carry += tot;
    }
    if (threadIdx.x == 0) *total = carry;
}

// K consecutive elements at a 16-byte aligned address, as 16-byte accesses.
template <class T, int K>
__device__ __forceinline__ void load_run16(const T* p, T (&v)[K])
{
    static_assert((sizeof(T) * K) % 16 == 0, "whole 16-byte words");
    const uint4* q = reinterpret_cast<const uint4*>(p);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) * K / 16); i++) {
        const uint4 u = q[i];
        memcpy(reinterpret_cast<char*>(v) + 16 * i, &u, 16);
    }
}

template <class T, int K>
__device__ __forceinline__ void store_run16(T* p, const T (&v)[K])
{
    static_assert((sizeof(T) * K) % 16 == 0, "whole 16-byte words");
    uint4* q = reinterpret_cast<uint4*>(p);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(T) * K / 16); i++) {
        uint4 u;
        memcpy(&u, reinterpret_cast<const char*>(v) + 16 * i, 16);
        q[i] = u;
    }
}

// kScanTile / kBS consecutive elements from `base` per thread of a workgroup
// of BS, scanned from `before`; returns the workgroup's sum.  Read and written
// as 16-byte accesses when the run is whole and both arrays are 16-byte
// aligned (the run starts at a multiple of its length, at least 32 bytes).
template <int BS, class TI, class TO, class Ld>
__device__ __forceinline__ TO scan_run(const TI* in, TO* out, int64_t n, int64_t base, TO before, TO* lds, Ld ld)
{
    constexpr int IPT = kScanTile / kBS;
    const bool vec = base + IPT <= n &&
                     ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    TO v[IPT];
    TO s = 0;
    if (vec) {
        TI r[IPT];
        load_run16(in + base, r);
#pragma unroll
        for (int k = 0; k < IPT; k++) v[k] = (TO)ld(r[k]);
    } else {
#pragma unroll
        for (int k = 0; k < IPT; k++) {
            const int64_t i = base + k;
            v[k] = i < n ? (TO)ld(in[i]) : TO(0);
        }
    }
#pragma unroll
    for (int k = 0; k < IPT; k++) s += v[k];
    if constexpr (std::is_same<Ld, LoadBlocks>::value) ld.template sums<IPT>(base, n, s);
    TO tot;
    TO ex = ftd::block_excl_scan<TO, BS>(s, lds, &tot) + before;
    if (vec) {
        TO o[IPT];
#pragma unroll
        for (int k = 0; k < IPT; k++) {
            o[k] = ex;
            ex += v[k];
        }
        store_run16(out + base, o);
    } else {
#pragma unroll
        for (int k = 0; k < IPT; k++) {
            const int64_t i = base + k;
            if (i < n) out[i] = ex;
            ex += v[k];
        }
    }
    if (Ld::clear)
        for (int k = 0; k < IPT; k++)
            if (base + k < n) const_cast<TI*>(in)[base + k] = TI(0);
    return tot;
}

template <class TI, class TO, class Ld>
__global__ __launch_bounds__(kBS) void k_scan_down(const TI* in, TO* out, int64_t n,
                                                   const TO* bsum, Ld ld)
{
    __shared__ TO lds[kBS / 64 + 1];
    scan_run<kBS>(in, out, n, (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * (kScanTile / kBS),
                  bsum[blockIdx.x], lds, ld);
}

// A short scan in one launch, by one workgroup, instead of three: small
// reinits are bound by their launches (32^3 points 305 us with three launches a
// scan, 256 with one; 47 x 33 x 17 triangles 503 and 466), and up to one step
// of the workgroup the scan itself is no slower.  With 32768 elements (four
// steps) a 127^3 reinit loses 25 us of 1320 to the longer scans.
constexpr int64_t kScanOne = 8192;
template <class TI, class TO, class Ld>
__global__ __launch_bounds__(1024) void k_scan_one(const TI* in, TO* out, int64_t n, TO* total, Ld ld)
{
    __shared__ TO lds[1024 / 64 + 1];
    constexpr int IPT = kScanTile / kBS;
    TO carry = TO(0);
    for (int64_t at = 0; at < n; at += 1024 * IPT)
        carry += scan_run<1024>(in, out, n, at + (int64_t)threadIdx.x * IPT, carry, lds, ld);
    if (threadIdx.x == 0) *total = carry;
}

// ============================================================================
// Mesh set-up: Morton order of the nodes (processing order of k_query)
// ============================================================================
// Fields: a handle holds one or more independent fields (a plain reinit has
// one).  Field k owns nodes [node_off[k], node_off[k+1]) and likewise tets and
// edges; its index bins and query tiles never mix with another field's.
// Node sort of one field (nodes node_base.. of xyz, local index i).
__global__ __launch_bounds__(kBS) void k_node_bin(const float* xyz, int64_t n, Grid g,
                                                  uint32_t* code, uint32_t* count)
{
    const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (i >= n) return;
    const uint32_t c = ftd::grid_code(g, xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2]);
    code[i] = c;
    atomicAdd(&count[c], 1u);
}

// Local node i to its query slot: its place in the sorted order, or, with
// cpb > 0, in its block's tiles (block_tile: the tiles before each block).
// cap: the field's slots; a node past them is left out and flagged.  The bins'
// counts are zero again at the end.
__global__ __launch_bounds__(kBS) void k_node_scatter(const float* xyz, int64_t n, int64_t node_base,
                                                      const uint32_t* code, uint32_t* count,
                                                      const uint32_t* offset, int cpb, const uint32_t* block_tile,
                                                      int64_t cap, unsigned long long* misfit, int32_t* perm,
                                                      float* sx, float* sy, float* sz)
{
    const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (i >= n) return;
    const uint32_t c = code[i];
    int64_t slot = (int64_t)offset[c] + atomicSub(&count[c], 1u) - 1u;
    if (cpb) {
        const uint32_t b = c / (uint32_t)cpb;
        slot += 64 * (int64_t)block_tile[b] - (int64_t)offset[b * (uint32_t)cpb];
    }
    if (slot >= cap) {
        *misfit = 1ull;
        return;
    }
    perm[slot] = (int32_t)(node_base + i);
    sx[slot] = xyz[3 * i];
    sy[slot] = xyz[3 * i + 1];
    sz[slot] = xyz[3 * i + 2];
}

// Padding slots (perm -1): coordinates of their tile's first slot, a node
// (lanes that only shadow it); tile -> field table.
__global__ __launch_bounds__(kBS) void k_pad_slots(int64_t n_slots, int nf, const int64_t* slot_off, const int32_t* perm,
                                                   float* sx, float* sy, float* sz, int32_t* tile_field,
                                                   unsigned long long* misfit)
{
    const int64_t s = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (s >= n_slots) return;
    const int64_t t0 = s & ~(int64_t)63;
    if (s == t0) tile_field[s >> 6] = ftd::field_of(slot_off, nf, s);
    if (perm[s] >= 0) return;
    if (perm[t0] < 0) {                                // a tile without nodes: fewer blocks than expected
        *misfit = 1ull;
        return;
    }
    sx[s] = sx[t0];
    sy[s] = sy[t0];
    sz[s] = sz[t0];
}

// ============================================================================
// Marching tets (LevelSet::findInterfaceNodes_ / reconstructInterface_)
// ============================================================================
// Opens a reinit: the nodes' signs, and everything that the stages mark or
// raise cleared.
__global__ __launch_bounds__(kBS) void k_node_signs(const double* phi, int64_t n, uint64_t* bits, uint64_t* retain,
                                                    uint64_t* ebits, int64_t nw_edges, uint64_t* sc)
{
    const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
    for (int64_t w = i; w < nw_edges; w += (int64_t)gridDim.x * kBS) ebits[w] = 0ull;
    if (i == 0) {
        sc[S_ERR] = ~0ull;
        sc[S_CAP] = 0ull;
        sc[S_EDGES] = 0ull;                            // the edge scan writes the low 32 bits
    }
    const int neg = (i < n) ? ftd::sign_bit(phi[i]) : 0;   // std::signbit (LevelSet.cpp:281,380)
    const uint64_t m = __ballot(neg);
    if (ftd::lane_id() == 0 && i < n) {
        bits[i >> 6] = m;
        retain[i >> 6] = 0ull;
    }
}

// Crossing iff 1..3 of a tet's nodes are negative (LevelSet.cpp:380-383); 2
// negative nodes -> 4 crossing edges -> 2 triangles.  A workgroup handles
// kClassifyGroups consecutive groups of kBS tets, one tet of each per
// thread, so that each thread has that many tet loads in flight; per group
// it writes the words of two bitmaps, crossing tets (tbits) and those with
// two triangles (t2bits, a subset), and blk[group] = (crossing tets << 32) |
// triangles.
constexpr int kClassifyGroups = 2;
__global__ __launch_bounds__(kBS) void k_classify(MeshView mv, int64_t T,
                                                  const uint64_t* sbits, uint64_t* tbits,
                                                  uint64_t* t2bits, uint64_t* blk)
{
    __shared__ uint64_t part[kClassifyGroups][kBS / 64];
    __shared__ int kf0;
    int4 q[kClassifyGroups];
    int64_t t[kClassifyGroups];
    // per-field arrays: the block's first field by binary search, then each
    // thread steps forward over the few field ends inside the block
    int k = 0;
    if (!mv.tets) {
        if (threadIdx.x == 0) kf0 = mv_tet_field(mv, std::min<int64_t>(T - 1, (int64_t)blockIdx.x * kClassifyGroups * kBS));
        __syncthreads();
        k = kf0;
    }
#pragma unroll
    for (int g = 0; g < kClassifyGroups; g++) {
        t[g] = ((int64_t)blockIdx.x * kClassifyGroups + g) * kBS + threadIdx.x;
        if (t[g] < T) {
            if (!mv.tets)
                while (t[g] >= mv.tet_off[k + 1]) k++;
            q[g] = mv_tet(mv, t[g], k);
        }
    }
#pragma unroll
    for (int g = 0; g < kClassifyGroups; g++) {
        int sgn = 0;
        if (t[g] < T)
            sgn = ftd::get_bit(sbits, q[g].x) + ftd::get_bit(sbits, q[g].y) + ftd::get_bit(sbits, q[g].z) +
                  ftd::get_bit(sbits, q[g].w);
        const bool cross = (t[g] < T) && sgn != 0 && sgn != 4;
        const uint64_t m = __ballot(cross);
        const uint64_t m2 = __ballot(cross && sgn == 2);
        if (ftd::lane_id() == 0 && t[g] < T) {
            tbits[t[g] >> 6] = m;
            t2bits[t[g] >> 6] = m2;
        }
        if (ftd::lane_id() == 0)
            part[g][threadIdx.x / 64] = ((uint64_t)__popcll(m) << 32) | (uint64_t)(__popcll(m) + __popcll(m2));
    }
    __syncthreads();
    if (threadIdx.x < kClassifyGroups) {
        const int64_t grp = (int64_t)blockIdx.x * kClassifyGroups + threadIdx.x;
        if (grp * kBS < T) {
            uint64_t s4 = 0;
            for (int w = 0; w < kBS / 64; w++) s4 += part[threadIdx.x][w];
            blk[grp] = s4;
        }
    }
}

// Capacities of a reinit whose buffers were sized in advance (graph replay; a
// negative one is not checked).  The first kernel that writes what a stage total
// counts compares the two in every thread, writes nothing when the total is
// larger, and raises S_CAP, which halts every later kernel.
__device__ __forceinline__ bool outgrown(uint64_t* sc, bool larger, uint64_t bit)
{
    if (larger && blockIdx.x == 0 && threadIdx.x == 0) sc[S_CAP] |= bit;
    return larger;
}

// One thread per 64-tet word of the crossing bitmap.  Lanes 4k..4k+3 share a
// k_classify block, whose exclusive offset is blk_prefix[w/4].
__global__ __launch_bounds__(kBS) void k_compact(const uint64_t* tbits, const uint64_t* t2bits,
                                                 int64_t nwords, const uint64_t* blk_prefix,
                                                 int32_t* xtet, int32_t* xtri_off, uint64_t* sc,
                                                 int64_t x_cap, int64_t f_cap)
{
    if (halted(sc) || outgrown(sc, x_cap >= 0 && (cnt_xtets(sc) > x_cap || cnt_tris(sc) > f_cap), 1ull)) return;
    const int64_t w = (int64_t)blockIdx.x * kBS + threadIdx.x;
    const uint64_t word = w < nwords ? tbits[w] : 0ull;
    const uint64_t two = w < nwords ? t2bits[w] : 0ull;
    const uint32_t ct = (uint32_t)(__popcll(word) + __popcll(two));
    const uint64_t mine = ((uint64_t)__popcll(word) << 32) | ct;
    uint64_t inc = mine;
#pragma unroll
    for (int o = 1; o < 4; o <<= 1) {
        const uint64_t t = ftd::shfl_up_u64(inc, o, 4);
        if ((int)(threadIdx.x & 3) >= o) inc += t;
    }
    if (w >= nwords || word == 0) return;
    const uint64_t base = blk_prefix[w >> 2] + (inc - mine);
    uint32_t bx = (uint32_t)(base >> 32), bt = (uint32_t)base;
    uint64_t m = word;
    while (m) {
        const int b = __ffsll((unsigned long long)m) - 1;
        m &= m - 1;
        xtet[bx] = (int32_t)(w * 64 + b);
        xtri_off[bx] = (int32_t)bt;
        bx++;
        bt += 1u + (uint32_t)((two >> b) & 1ull);
    }
}

// Error word: (code << 40) | tet, min-reduced so the lowest failing tet wins
// within a code; codes: 1 = t2e (FT_ERR_T2E), 2 = degenerate tet.
__device__ __forceinline__ void flag_error(unsigned long long* err, int code, int64_t t)
{
    atomicMin(err, ((unsigned long long)code << 40) | (unsigned long long)t);
}

// Bit i of a bitmap that many set at once: no atomic where it is already set
// (as seen by all of the device).
__device__ __forceinline__ void set_bit(unsigned long long* bits, int64_t i)
{
    const unsigned long long m = 1ull << (i & 63);
    if (!(__hip_atomic_load(&bits[i >> 6], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & m)) atomicOr(&bits[i >> 6], m);
}

// Crossing tets: collect crossing edges in t2e order (LevelSet.cpp:385-391),
// check the count (3 or 4, and consistent with the node signs used for the
// triangle offsets: 4 exactly for the tets of the two-triangle bitmap t2bits),
// mark them in the edge bitmap (each edge is marked by about six tets, and the
// marks bound it: at 256^3, 0.92M crossing tets, 149 us with an atomic each, now
// 92).
__global__ __launch_bounds__(kBS) void k_xtet(const uint64_t* t2bits, MeshView mv,
                                              const uint64_t* sbits,
                                              const int32_t* xtet, uint64_t* sc,
                                              unsigned long long* ebits, int4* xedges)
{
    if (halted(sc)) return;
    const int64_t x = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (x >= cnt_xtets(sc)) return;
    unsigned long long* err = (unsigned long long*)(sc + S_ERR);
    const int64_t t = xtet[x];
    const int k = mv.t2e3 ? 0 : mv_tet_field(mv, t);
    const int2 r0 = mv_t2e(mv, t, 0, k), r1 = mv_t2e(mv, t, 1, k), r2 = mv_t2e(mv, t, 2, k);
    const int te[6] = {r0.x, r0.y, r1.x, r1.y, r2.x, r2.y};
    int ce[4] = {-1, -1, -1, -1};
    int n = 0;
#pragma unroll
    for (int j = 0; j < 6; j++) {
        const int2 ab = mv_edge(mv, te[j], k);          // a tet's edges are its field's
        if (ftd::get_bit(sbits, ab.x) != ftd::get_bit(sbits, ab.y)) {
            if (n < 4) ce[n] = te[j];
            n++;
        }
    }
    const int expect = ftd::get_bit(t2bits, t) ? 4 : 3;
    if (n != expect) {
        flag_error(err, 1, t);
        xedges[x] = make_int4(-1, -1, -1, -1);
        return;
    }
    for (int k = 0; k < n; k++) set_bit(ebits, ce[k]);
    xedges[x] = make_int4(ce[0], ce[1], ce[2], ce[3]);
}

__device__ __forceinline__ int32_t edge_rank(const uint64_t* ebits, const uint32_t* eprefix,
                                             int32_t e)
{
    const uint64_t wv = ebits[e >> 6];
    const uint64_t below = (e & 63) ? (wv & ((1ull << (e & 63)) - 1ull)) : 0ull;
    return (int32_t)(eprefix[e >> 6] + (uint32_t)__popcll(below));
}

// Position of the n-th (from 0) set bit of w; n < popcount(w).
__device__ __forceinline__ int nth_set_bit(uint64_t w, uint32_t n)
{
    int pos = 0;
#pragma unroll
    for (int sh = 32; sh; sh >>= 1) {
        const uint32_t c = (uint32_t)__popcll(w & ((1ull << sh) - 1ull));
        const bool skip = n >= c;
        n -= skip ? c : 0u;
        w = skip ? (w >> sh) : w;
        pos += skip ? sh : 0;
    }
    return pos;
}

// Crossing points in increasing edge order (LevelSet.cpp:278-299).  A wave
// takes 64 consecutive words of the edge bitmap and their crossing edges 64
// at a time, one per lane: the lane finds the word holding its edge by a
// binary search over the wave's prefix counts, then the bit.  FP64
// interpolation, no fma; marks both edge nodes as retained
// (LevelSet.cpp:443-447).
__global__ __launch_bounds__(kBS) void k_points(const uint64_t* ebits, const uint32_t* eprefix,
                                                int64_t nwords, MeshView mv,
                                                const float* xyz, const double* phi,
                                                float* ifp, int32_t* ifp2e,
                                                unsigned long long* retain, uint64_t* sc, int64_t p_cap)
{
    if (halted(sc) || outgrown(sc, p_cap >= 0 && cnt_points(sc) > p_cap, 2ull)) return;
    const int lane = ftd::lane_id();
    const int64_t w = (int64_t)blockIdx.x * kBS + threadIdx.x;
    const int64_t w0 = w - lane;                       // the wave's first word
    if (w0 >= nwords) return;                          // whole wave out of range
    const uint64_t word = w < nwords ? ebits[w] : 0ull;
    const uint32_t cnt = (uint32_t)__popcll(word);
    const uint32_t inc = ftd::wave_incl_scan(cnt);
    const uint32_t total = __shfl(inc, 63);
    const uint32_t r0 = eprefix[w0];                   // rank of the wave's first crossing edge
    for (uint32_t k0 = 0; k0 < total; k0 += 64) {
        const uint32_t k = k0 + lane;
        int L = 0;                                     // lanes whose words end at or before k
#pragma unroll
        for (int step = 32; step; step >>= 1) {
            const uint32_t v = __shfl(inc, L + step - 1);
            L += (v <= k) ? step : 0;
        }
        const uint64_t wl = __shfl(word, L);
        const uint32_t ex = __shfl(inc, L) - __shfl(cnt, L);
        if (k >= total) continue;
        const int64_t e = (w0 + L) * 64 + nth_set_bit(wl, k - ex);
        const uint32_t r = r0 + k;
        const int2 ab = mv_edge(mv, e, mv.edges ? 0 : mv_edge_field(mv, e));
        const double pa = phi[ab.x], pb = phi[ab.y];
        double t = 0.5;
        const double div = pa - pb;
        if (fabs(div) > (double)FLT_MIN) t = pa / div;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const double p0 = (double)xyz[3 * (int64_t)ab.x + c];
            const double p1 = (double)xyz[3 * (int64_t)ab.y + c];
            const double v = (1.0 - t) * p0 + t * p1;
            ifp[3 * (int64_t)r + c] = (float)v;
        }
        ifp2e[r] = (int32_t)e;
        atomicOr(&retain[ab.x >> 6], 1ull << (ab.x & 63));
        atomicOr(&retain[ab.y >> 6], 1ull << (ab.y & 63));
    }
}

// addTriangle (LevelSet.cpp:330-357): float normal by Eigen's cross product,
// orientation toward phi > 0 through the first tet node with |phi| > FLT_MIN.
__device__ __forceinline__ void emit_tri(int32_t n0, int32_t n1, int32_t n2, int32_t pref,
                                         const float* xyz, const double* phi, const float* ifp,
                                         int32_t f, int4* tris, float* tri_norm)
{
    const float* q0 = ifp + 3 * (int64_t)n0;
    const float* q1 = ifp + 3 * (int64_t)n1;
    const float* q2 = ifp + 3 * (int64_t)n2;
    const float e1x = q1[0] - q0[0], e1y = q1[1] - q0[1], e1z = q1[2] - q0[2];
    const float e2x = q2[0] - q0[0], e2y = q2[1] - q0[1], e2z = q2[2] - q0[2];
    const float nx = e1y * e2z - e1z * e2y;
    const float ny = e1z * e2x - e1x * e2z;
    const float nz = e1x * e2y - e1y * e2x;
    const float* pr = xyz + 3 * (int64_t)pref;
    const float rx = pr[0] - q0[0], ry = pr[1] - q0[1], rz = pr[2] - q0[2];
    const float dot = nx * rx + (ny * ry + nz * rz);     // Eigen redux: x0 + (x1 + x2)
    const int sd = (int)(__float_as_uint(dot) >> 31);
    int4 out;
    out.x = n0;
    if (sd != ftd::sign_bit(phi[pref])) { out.y = n2; out.z = n1; }
    else { out.y = n1; out.z = n2; }
    out.w = -1;
    tris[f] = out;
    const float sq = nx * nx + (ny * ny + nz * nz);
    tri_norm[f] = sqrtf(sq);
}

__global__ __launch_bounds__(kBS) void k_tris(MeshView mv, const float* xyz,
                                              const double* phi, const int32_t* xtet,
                                              const int32_t* xtri_off, const int4* xedges,
                                              const uint64_t* ebits,
                                              const uint32_t* eprefix, const float* ifp,
                                              int4* tris, float* tri_norm, int32_t* if_elems,
                                              uint64_t* sc)
{
    if (halted(sc)) return;
    const int64_t x = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (x >= cnt_xtets(sc)) return;
    unsigned long long* err = (unsigned long long*)(sc + S_ERR);
    const int64_t t = xtet[x];
    if_elems[x] = (int32_t)t;
    const int4 ce = xedges[x];
    if (ce.x < 0) return;                                  // flagged by k_xtet
    const int4 q = mv_tet(mv, t, mv.tets ? 0 : mv_tet_field(mv, t));
    const int nd[4] = {q.x, q.y, q.z, q.w};
    int k = 0;
    while (k < 4 && fabs(phi[nd[k]]) <= (double)FLT_MIN) k++;
    if (k == 4) { flag_error(err, 2, t); return; }
    const int32_t pref = nd[k];
    const int32_t v0 = edge_rank(ebits, eprefix, ce.x);
    const int32_t v1 = edge_rank(ebits, eprefix, ce.y);
    const int32_t v2 = edge_rank(ebits, eprefix, ce.z);
    const int32_t f = xtri_off[x];
    if (ce.w < 0) {
        emit_tri(v0, v1, v2, pref, xyz, phi, ifp, f, tris, tri_norm);          // :393-395
    } else {
        const int32_t v3 = edge_rank(ebits, eprefix, ce.w);
        emit_tri(v0, v2, v3, pref, xyz, phi, ifp, f, tris, tri_norm);          // :397
        emit_tri(v0, v1, v3, pref, xyz, phi, ifp, f + 1, tris, tri_norm);      // :398
    }
}

// Point -> triangle lists and point areas; the per-element steps, with their
// index checks, are in ft_p2t.hpp.
struct AtomicInc {
    __device__ uint32_t operator()(uint32_t* p) const { return atomicAdd(p, 1u); }
};

__global__ __launch_bounds__(kBS) void k_p2t_count(const int4* tris, uint64_t* sc, uint32_t* deg)
{
    if (halted(sc)) return;
    const int64_t f = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (f >= cnt_tris(sc)) return;
    const int4 t = tris[f];
    const int32_t v[3] = {t.x, t.y, t.z};
    if (!ftp::count_tri(v, cnt_points(sc), deg, AtomicInc{}))
        flag_error((unsigned long long*)(sc + S_ERR), ftp::kErrIndex, f);
}

__global__ __launch_bounds__(kBS) void k_p2t_fill(const int4* tris, uint64_t* sc,
                                                  const uint32_t* off, uint32_t* cursor,
                                                  int32_t* p2t)
{
    if (halted(sc)) return;
    const int64_t f = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (f >= cnt_tris(sc)) return;
    const int4 t = tris[f];
    const int32_t v[3] = {t.x, t.y, t.z};
    if (!ftp::fill_tri(v, (int32_t)f, cnt_points(sc), off, cursor, p2t, AtomicInc{}))
        flag_error((unsigned long long*)(sc + S_ERR), ftp::kErrIndex, f);
}

__global__ __launch_bounds__(kBS) void k_point_area(const uint32_t* off, uint64_t* sc,
                                                    int32_t* p2t, const float* tri_norm,
                                                    float* area)
{
    if (halted(sc)) return;
    const int64_t v = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (v >= cnt_points(sc)) return;
    if (!ftp::point_area(v, off, p2t, cnt_tris(sc), tri_norm, area))
        flag_error((unsigned long long*)(sc + S_ERR), ftp::kErrIndex, v);
}

// ============================================================================
// Spatial index: uniform bins as a bitmap, 64-ary tree of oriented boxes
// ============================================================================
// The bins of a field are numbered along the Morton curve, one bit each.  A
// 64-bit word of the bitmap is then a 4 x 4 x 4 block of bins, and words of
// words are the larger blocks: the tree has one node per non-empty block and
// its children (at most 64) are consecutive in the Morton order of the
// non-empty bins.  Leaves (non-empty bins) and nodes of all levels share one
// numbering, level by level (LevelOff), so first[g], first[g + 1] is a
// node's range of children, or a leaf's range of primitives.
//
// Nothing here grows with the bins but the bitmap and its prefix (12 bytes
// per 64 bins): at 256^3, 2^24 bins, clearing, scanning and compacting
// one counter per bin took 0.30 ms of a reinit; the bitmap's take 0.03 ms.
constexpr int kNodeBlocks = 2048;            // workgroups of a node level (waves take nodes in turn)
constexpr int kLevels = 5;                   // leaves and 4 levels of nodes (2^24 bins per field)

struct LevelOff {
    uint32_t off[kLevels];                   // first index of each level
};

// Bounding volume of a primitive, a leaf or a node as the search reads it: a
// box with unit axes x, y, z and half extents e, in the field's scaled
// coordinates p' = (p - org) inv_s.  Row k = (axis, offset) applied to (p', 1)
// is p's coordinate along axis k from the box centre, so four boxes are 16
// rows (the fourth of each, its extents, is a spare one) of a 16 x 16 matrix
// product and 16 nodes its columns.
//
// A row is kept as eight halves (axis, offset) + (axis, offset): each value
// is the sum of its nearest half and the half of what is left, 22 bits, and
// the node's coordinates are split the same way.  The 16 terms of a row's
// product are then exact in the f16 matrix instruction's FP32 sum, which
// leaves 2^-22.8 of a scaled unit at most (measured over random boxes and
// nodes; 2^-23.9 for the FP32 instruction); the search allows 2^-20.  The FP32
// instruction 16x16x4 holds the vector unit for its 32 cycles (4 of them and
// 32 fma: 290 cycles per wave on a full SIMD, 136 and 138 each alone); the f16
// 16x16x16 runs beside it (153 cycles with the same 32 fma).
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
struct __align__(16) Row {
    v4h hi, lo;
};
struct __align__(16) Item {
    Row x, y, z;
    float4 e;                                // half extents (scaled), 0
};
__device__ __forceinline__ Row make_row(float x, float y, float z, float w)
{
    Row r;
    r.hi = v4h{(_Float16)x, (_Float16)y, (_Float16)z, (_Float16)w};
    r.lo = v4h{(_Float16)(x - (float)r.hi[0]), (_Float16)(y - (float)r.hi[1]), (_Float16)(z - (float)r.hi[2]),
               (_Float16)(w - (float)r.hi[3])};
    return r;
}
__device__ __forceinline__ float4 row_values(const Row& r)
{
    return make_float4((float)r.hi[0] + (float)r.lo[0], (float)r.hi[1] + (float)r.lo[1],
                       (float)r.hi[2] + (float)r.lo[2], (float)r.hi[3] + (float)r.lo[3]);
}
// The item that admits every point.
__device__ __forceinline__ Item open_item()
{
    Item it;
    it.x = it.y = it.z = make_row(0.0f, 0.0f, 0.0f, 0.0f);
    it.e = make_float4(1e30f, 1e30f, 1e30f, 0.0f);
    return it;
}

__device__ __forceinline__ void tri_vertices(const int4* tris, const float* ifp, int32_t f,
                                             float* a, float* b, float* c)
{
    const int4 t = tris[f];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        a[k] = ifp[3 * (int64_t)t.x + k];
        b[k] = ifp[3 * (int64_t)t.y + k];
        c[k] = ifp[3 * (int64_t)t.z + k];
    }
}

// Index geometry of one reinit: per-field grids and bin offsets (multiples
// of 64), the field of a crossing point through its edge (edge_off).
struct IndexGeom {
    const int64_t* edge_off;         // nf + 1
    const int64_t* cnt_off;          // nf + 1
    const Grid* grids;               // nf
    int nf;
};
__device__ __forceinline__ int bin_field(const IndexGeom& ig, uint32_t c)
{
    return ig.nf > 1 ? ftd::field_of(ig.cnt_off, ig.nf, (int64_t)c) : 0;
}

// mode 0: points (ifp), mode 1: triangles (centroid).
__device__ __forceinline__ int64_t cnt_prims(int mode, const uint64_t* sc)
{
    return mode == 0 ? cnt_points(sc) : cnt_tris(sc);
}

// The run of lanes around this one that hold the same v (lanes that returned
// are the wave's last): its first lane, and the lane after its last.
__device__ __forceinline__ void lane_run(uint32_t v, int& first, int& end)
{
    const int lane = ftd::lane_id();
    const int lanes = (int)__popcll(__ballot(true));   // (with every lane: not in the choice below)
    const uint32_t before = (uint32_t)__shfl_up((int)v, 1);
    const uint64_t heads = __ballot(lane == 0 || before != v), upto = ~0ull >> (63 - lane);
    first = 63 - __clzll((long long)(heads & upto));
    const uint64_t later = heads & ~upto;
    end = later ? __ffsll((unsigned long long)later) - 1 : lanes;
}

// Bin of each primitive, marked in the bitmap.  Neighbouring primitives often
// share their bin: the first lane of a run marks it, and needs no atomic where
// the word already holds the bit.  The atomics bound it and k_prim_rank: at
// 256^3 (1.2M triangles) 111 and 58 us with every lane on its own, now 55 and
// 20; 0.6M points 79 and 34, now 36 and 12.  (That is without the point lists
// beside them: while k_p2t_count and k_p2t_fill run on the side stream both
// take 80 to 105 us in some calls.)
__global__ __launch_bounds__(kBS) void k_prim_bin(int mode, const uint64_t* sc, const float* ifp,
                                                  const int4* tris, const int32_t* ifp2e,
                                                  IndexGeom ig, uint32_t* code, unsigned long long* bits)
{
    if (halted(sc)) return;
    const int64_t j = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (j >= cnt_prims(mode, sc)) return;
    float c[3];
    int32_t v0;
    if (mode == 0) {
        for (int k = 0; k < 3; k++) c[k] = ifp[3 * j + k];
        v0 = (int32_t)j;
    } else {
        float a[3], b[3], d[3];
        tri_vertices(tris, ifp, (int32_t)j, a, b, d);
        for (int k = 0; k < 3; k++) c[k] = (a[k] + b[k] + d[k]) * (1.0f / 3.0f);
        v0 = tris[j].x;
    }
    const int f = ifp2e ? ftd::field_of(ig.edge_off, ig.nf, ifp2e[v0]) : 0;
    const uint32_t cc = (uint32_t)ig.cnt_off[f] + ftd::grid_code(ig.grids[f], c[0], c[1], c[2]);
    code[j] = cc;
    int first, end;
    lane_run(cc, first, end);
    if (first != ftd::lane_id()) return;
    set_bit(bits, cc);
}

// Leaf of each primitive (the rank of its bin's bit) and its place among the
// leaf's primitives (a run of lanes with one leaf takes its places together);
// code becomes the leaf.
__global__ __launch_bounds__(kBS) void k_prim_rank(int mode, const uint64_t* sc, const uint64_t* bits,
                                                   const uint32_t* wprefix, uint32_t* code, uint32_t* place,
                                                   uint32_t* leaf_cnt, uint32_t* leaf_bin)
{
    if (halted(sc)) return;
    const int64_t j = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (j >= cnt_prims(mode, sc)) return;
    const uint32_t c = code[j];
    const uint64_t below = bits[c >> 6] & ((1ull << (c & 63)) - 1ull);
    const uint32_t l = wprefix[c >> 6] + (uint32_t)__popcll(below);
    code[j] = l;
    int first, end;
    lane_run(l, first, end);
    uint32_t at = 0;
    if (first == ftd::lane_id()) {
        at = atomicAdd(&leaf_cnt[l], (uint32_t)(end - first));
        leaf_bin[l] = c;                         // the same value from each of its primitives
    }
    place[j] = (uint32_t)__shfl((int)at, first) + (uint32_t)(ftd::lane_id() - first);
}

// What leaf l adds to the level scan: its primitives, and 1 for each level
// at which it opens a new node (its bin's code differs from the previous
// leaf's above that level's bits, or the field does).
__device__ __forceinline__ ftd::Lv leaf_elem(int64_t l, int64_t L, const uint32_t* leaf_cnt,
                                             const uint32_t* leaf_bin, const IndexGeom& ig, uint32_t* opens,
                                             int* field)
{
    *opens = 0u;
    *field = 0;
    if (l >= L) return ftd::Lv(0);
    const uint32_t c = leaf_bin[l];
    const int f = bin_field(ig, c);
    const uint32_t f0 = (uint32_t)ig.cnt_off[f];
    const uint32_t p = l > 0 ? leaf_bin[l - 1] : 0u;
    uint32_t o = 31u;                            // bit 4: the field's first leaf
    if (l > 0 && p >= f0) {
        const uint32_t x = (p - f0) ^ (c - f0);
        o = ((x >> 6) ? 1u : 0u) | ((x >> 12) ? 2u : 0u) | ((x >> 18) ? 4u : 0u) | ((x >> 24) ? 8u : 0u);
    }
    *opens = o;
    *field = f;
    ftd::Lv v;
    v.a = (uint64_t)leaf_cnt[l] | ((uint64_t)(o & 1u) << 32);
    v.b = (uint64_t)((o >> 1) & 1u) | ((uint64_t)((o >> 2) & 1u) << 32);
    v.c = (uint64_t)((o >> 3) & 1u);
    return v;
}

__global__ __launch_bounds__(kBS) void k_level_reduce(const uint64_t* sc, const uint32_t* leaf_cnt,
                                                      const uint32_t* leaf_bin, IndexGeom ig, ftd::Lv* bsum)
{
    __shared__ ftd::Lv lds[kBS / 64 + 1];
    const int64_t L = halted(sc) ? 0 : cnt_leaves(sc);
    const int64_t base = (int64_t)blockIdx.x * kScanTile;
    ftd::Lv s(0);
    if (base < L)
        for (int k = 0; k < kScanTile / kBS; k++) {
            uint32_t o;
            int f;
            s += leaf_elem(base + (int64_t)k * kBS + threadIdx.x, L, leaf_cnt, leaf_bin, ig, &o, &f);
        }
    ftd::Lv tot;
    ftd::block_excl_scan<ftd::Lv, kBS>(s, lds, &tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// first[] of the leaves and of the nodes of every level, and the fields'
// roots: the node of the level that covers the whole field (Grid::root_lv).
// IPT leaves from `base` per thread of a workgroup of BS, after `before`;
// returns the workgroup's sum.
template <int BS, int IPT>
__device__ __forceinline__ ftd::Lv level_run(int64_t base, int64_t L, const uint32_t* leaf_cnt,
                                             const uint32_t* leaf_bin, const IndexGeom& ig, ftd::Lv before,
                                             const LevelOff& lo, uint32_t* first, uint32_t* roots, ftd::Lv* lds)
{
    ftd::Lv s(0);
    for (int k = 0; k < IPT; k++) {
        uint32_t o;
        int f;
        s += leaf_elem(base + k, L, leaf_cnt, leaf_bin, ig, &o, &f);
    }
    ftd::Lv tot;
    ftd::Lv ex = ftd::block_excl_scan<ftd::Lv, BS>(s, lds, &tot) + before;
    for (int k = 0; k < IPT; k++) {
        const int64_t l = base + k;
        if (l >= L) break;
        uint32_t o;
        int f;
        const ftd::Lv v = leaf_elem(l, L, leaf_cnt, leaf_bin, ig, &o, &f);
        // this leaf's node at each level, were it to open one
        uint32_t g[kLevels] = {(uint32_t)l, lo.off[1] + (uint32_t)(ex.a >> 32), lo.off[2] + (uint32_t)ex.b,
                               lo.off[3] + (uint32_t)(ex.b >> 32), lo.off[4] + (uint32_t)ex.c};
        first[l] = (uint32_t)ex.a;
#pragma unroll
        for (int q = 1; q < kLevels; q++)
            if ((o >> (q - 1)) & 1u) first[g[q]] = g[q - 1];
        if (o & 16u) {
            const int r = ig.grids[f].root_lv;
            roots[f] = r == 1 ? g[1] : r == 2 ? g[2] : r == 3 ? g[3] : g[4];
        }
        ex += v;
        if (l == L - 1) {                        // the ends of the last node of each level
            first[L] = (uint32_t)ex.a;
            first[lo.off[1] + (uint32_t)(ex.a >> 32)] = (uint32_t)L;
            first[lo.off[2] + (uint32_t)ex.b] = lo.off[1] + (uint32_t)(ex.a >> 32);
            first[lo.off[3] + (uint32_t)(ex.b >> 32)] = lo.off[2] + (uint32_t)ex.b;
            first[lo.off[4] + (uint32_t)ex.c] = lo.off[3] + (uint32_t)(ex.b >> 32);
        }
    }
    return tot;
}

__global__ __launch_bounds__(kBS) void k_level_down(const uint64_t* sc, const uint32_t* leaf_cnt,
                                                    const uint32_t* leaf_bin, IndexGeom ig, const ftd::Lv* bsum,
                                                    LevelOff lo, uint32_t* first, uint32_t* roots)
{
    __shared__ ftd::Lv lds[kBS / 64 + 1];
    constexpr int IPT = kScanTile / kBS;
    const int64_t L = halted(sc) ? 0 : cnt_leaves(sc);
    if ((int64_t)blockIdx.x * kScanTile >= L) return;            // whole block
    level_run<kBS, IPT>((int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * IPT, L, leaf_cnt, leaf_bin, ig,
                        bsum[blockIdx.x], lo, first, roots, lds);
}

// All of it for few leaves, in one launch by one workgroup (kScanOne's reason;
// the leaves are fewer than the bound on them that is compared: a bound of
// 32768 gives 10 us of 480 over 8192 at 47 x 33 x 17, 8 of 530 at 61^3 points).
constexpr int64_t kLevelOne = 32768;
constexpr int kLevelOneRun = 4;                        // leaves per thread and step
__global__ __launch_bounds__(1024) void k_level_one(uint64_t* sc, const uint32_t* leaf_cnt, const uint32_t* leaf_bin,
                                                    IndexGeom ig, LevelOff lo, uint32_t* first, uint32_t* roots)
{
    __shared__ ftd::Lv lds[1024 / 64 + 1];
    const int64_t L = halted(sc) ? 0 : cnt_leaves(sc);
    ftd::Lv carry(0);
    for (int64_t at = 0; at < L; at += 1024 * kLevelOneRun)
        carry += level_run<1024, kLevelOneRun>(at + (int64_t)threadIdx.x * kLevelOneRun, L, leaf_cnt, leaf_bin, ig,
                                               carry, lo, first, roots, lds);
    if (threadIdx.x == 0) *reinterpret_cast<ftd::Lv*>(sc + S_LV) = carry;
}

// The item of a box given by its axes, its centre m and half extents h in the
// mesh's coordinates.  The extents are rounded up by the error of a row's
// product (the search's own allowance covers centres within one scaled unit
// of the origin; farther ones, primitives outside the field's box, carry
// theirs here).  A box that is not finite admits every point.
__device__ __forceinline__ Item make_item(const Grid& g, const float ax[3][3], const double m[3], const float h[3])
{
    const double s = (double)g.inv_s;
    double mm[3], far2 = 0.0;
    for (int k = 0; k < 3; k++) {
        mm[k] = (m[k] - (double)g.org[k]) * s;
        far2 += mm[k] * mm[k];
    }
    Row r[3];
    float e[3];
    bool ok = far2 < 1e8;                              // offsets within the halves' range
    const float slack = 0x1.0p-22f + (far2 > 1.0 ? 0x1.0p-19f * sqrtf((float)far2) : 0.0f);
    for (int k = 0; k < 3; k++) {
        const double w = -((double)ax[k][0] * mm[0] + (double)ax[k][1] * mm[1] + (double)ax[k][2] * mm[2]);
        r[k] = make_row(ax[k][0], ax[k][1], ax[k][2], (float)w);
        e[k] = h[k] * g.inv_s * (1.0f + 0x1.0p-20f) + slack;
        ok = ok && fabsf(ax[k][0]) <= 2.0f && fabsf(ax[k][1]) <= 2.0f && fabsf(ax[k][2]) <= 2.0f && e[k] <= 1e15f;
    }
    if (!ok) return open_item();
    Item it;
    it.x = r[0]; it.y = r[1]; it.z = r[2];
    it.e = make_float4(e[0], e[1], e[2], 0.0f);
    return it;
}

// Scatter primitives into leaf order and write their search records.
__global__ __launch_bounds__(kBS) void k_prim_scatter(int mode, const uint64_t* sc, const float* ifp,
                                                      const int4* tris, const uint32_t* code,
                                                      const uint32_t* place, const uint32_t* first,
                                                      const uint32_t* leaf_bin, IndexGeom ig,
                                                      float4* prec, Item* titem, TriRec* trec, int32_t* pidx)
{
    if (halted(sc)) return;
    const int64_t j = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (j >= cnt_prims(mode, sc)) return;
    const uint32_t l = code[j];
    const uint32_t slot = first[l] + place[j];
    pidx[slot] = (int32_t)j;
    if (mode == 0) {
        prec[slot] = make_float4(ifp[3 * j], ifp[3 * j + 1], ifp[3 * j + 2], __int_as_float((int32_t)j));
        return;
    }
    float v3[3][3];
    tri_vertices(tris, ifp, (int32_t)j, v3[0], v3[1], v3[2]);
    // A triangle with a vertex that is not finite is nobody's nearest, not by its
    // other vertices' edge either: all its distances are NaN.
    bool finite = true;
    for (int q = 0; q < 3; q++)
        for (int k = 0; k < 3; k++) finite = finite && fabsf(v3[q][k]) < INFINITY;
    if (!finite)
        for (int q = 0; q < 3; q++)
            for (int k = 0; k < 3; k++) v3[q][k] = NAN;
    // Rotate (orientation kept) so that ab is the longest edge, then build the
    // frame in FP64: u along ab, n the unit normal, v = n x u.  Collinear or
    // coincident vertices get a frame along ab and no interior: the distance
    // is then that of the edge segments.
    double len[3];
    for (int q = 0; q < 3; q++) {
        const float* p0 = v3[q];
        const float* p1 = v3[(q + 1) % 3];
        double s = 0.0;
        for (int k = 0; k < 3; k++) { const double dd = (double)p1[k] - p0[k]; s += dd * dd; }
        len[q] = s;
    }
    const int r0 = (len[0] >= len[1] && len[0] >= len[2]) ? 0 : (len[1] >= len[2] ? 1 : 2);
    const float* a = v3[r0];
    const float* b = v3[(r0 + 1) % 3];
    const float* d = v3[(r0 + 2) % 3];
    double e0[3], e1[3];
    for (int k = 0; k < 3; k++) { e0[k] = (double)b[k] - a[k]; e1[k] = (double)d[k] - a[k]; }
    double nv[3];
    ftd::cross3d(e0, e1, nv);
    const double nn = ftd::dot3d(nv, nv);
    const double L0 = sqrt(ftd::dot3d(e0, e0));
    double u[3], v[3], nu[3];
    bool interior = nn > 0.0 && L0 > 0.0;
    if (L0 > 0.0) for (int k = 0; k < 3; k++) u[k] = e0[k] / L0;
    else { u[0] = 1.0; u[1] = 0.0; u[2] = 0.0; }
    if (interior) {
        const double inn = 1.0 / sqrt(nn);
        for (int k = 0; k < 3; k++) nu[k] = nv[k] * inn;
        ftd::cross3d(nu, u, v);
    } else {
        // any unit vector orthogonal to u
        const double t0[3] = {fabs(u[0]) < 0.9 ? 1.0 : 0.0, fabs(u[0]) < 0.9 ? 0.0 : 1.0, 0.0};
        double w[3];
        ftd::cross3d(u, t0, w);
        const double wl = sqrt(ftd::dot3d(w, w));
        for (int k = 0; k < 3; k++) v[k] = w[k] / wl;
        ftd::cross3d(u, v, nu);
    }
    const double Cx = ftd::dot3d(e1, u), Cy = interior ? ftd::dot3d(e1, v) : 0.0;
    const double dCx = Cx - L0;
    const double lac = Cx * Cx + Cy * Cy, lbc = dCx * dCx + Cy * Cy;
    TriRec r;
    r.a = make_float4(a[0], a[1], a[2], (float)dCx);
    r.u = make_float4((float)u[0], (float)u[1], (float)u[2], (float)L0);
    r.v = make_float4((float)v[0], (float)v[1], (float)v[2], (float)Cx);
    r.n = make_float4((float)nu[0], (float)nu[1], (float)nu[2], (float)Cy);
    r.i = make_float4(L0 > 0.0 ? (float)(1.0 / L0) : 0.0f, lac > 0.0 ? (float)(1.0 / lac) : 0.0f,
                      lbc > 0.0 ? (float)(1.0 / lbc) : 0.0f,
                      __int_as_float((int32_t)j | (interior ? 0 : INT32_MIN)));
    trec[slot] = r;
    if (!titem) return;
    // The rectangle [0, L0] x [0, Cy] of the frame holds the triangle: ab is
    // the longest edge, so C projects inside [0, L0], and Cy >= 0.
    const Grid& g = ig.grids[bin_field(ig, leaf_bin[l])];
    const double s = (double)g.inv_s;
    double m[3];
    for (int k = 0; k < 3; k++) m[k] = ((double)a[k] - (double)g.org[k] + 0.5 * (L0 * u[k] + Cy * v[k])) * s;
    Item it;
    it.x = make_row((float)u[0], (float)u[1], (float)u[2], (float)-ftd::dot3d(u, m));
    it.y = make_row((float)v[0], (float)v[1], (float)v[2], (float)-ftd::dot3d(v, m));
    it.z = make_row((float)nu[0], (float)nu[1], (float)nu[2], (float)-ftd::dot3d(nu, m));
    it.e = make_float4((float)(0.5 * L0 * s) * (1.0f + 0x1.0p-20f), (float)(0.5 * Cy * s) * (1.0f + 0x1.0p-20f), 0.0f,
                       0.0f);
    titem[slot] = it;
}

// Unit eigenvector of the smallest eigenvalue of the symmetric 3x3 matrix C
// (c00, c11, c22, c01, c02, c12): the eigenvalue in closed form (O. K. Smith,
// "Eigenvalues of a symmetric 3 x 3 matrix", CACM 4(4), 1961), the vector as
// the longest cross product of two rows of C - lambda I.  False when the
// points are (nearly) isotropic or there is no clear smallest direction.
__device__ inline bool smallest_eigvec(const double c[6], double n[3])
{
    const double p1 = c[3] * c[3] + c[4] * c[4] + c[5] * c[5];
    const double q = (c[0] + c[1] + c[2]) / 3.0;
    const double a = c[0] - q, b = c[1] - q, d = c[2] - q;
    const double p2 = a * a + b * b + d * d + 2.0 * p1;
    if (!(p2 > 0.0)) return false;
    const double p = sqrt(p2 / 6.0);
    const double B[6] = {a / p, b / p, d / p, c[3] / p, c[4] / p, c[5] / p};
    const double det = B[0] * (B[1] * B[2] - B[5] * B[5]) - B[3] * (B[3] * B[2] - B[5] * B[4]) +
                       B[4] * (B[3] * B[5] - B[1] * B[4]);
    const double r = fmin(1.0, fmax(-1.0, det / 2.0));
    const double lam = q + 2.0 * p * cos(acos(r) / 3.0 + 2.0943951023931957);   // smallest
    const double r0[3] = {c[0] - lam, c[3], c[4]}, r1[3] = {c[3], c[1] - lam, c[5]},
                 r2[3] = {c[4], c[5], c[2] - lam};
    double x[3][3];
    ftd::cross3d(r0, r1, x[0]);
    ftd::cross3d(r0, r2, x[1]);
    ftd::cross3d(r1, r2, x[2]);
    int best = 0;
    double bl = ftd::dot3d(x[0], x[0]);
    for (int k = 1; k < 3; k++) {
        const double lk = ftd::dot3d(x[k], x[k]);
        if (lk > bl) { bl = lk; best = k; }
    }
    if (!(bl > 1e-24 * p2 * p2)) return false;
    const double inv = 1.0 / sqrt(bl);
    for (int k = 0; k < 3; k++) n[k] = x[best][k] * inv;
    return true;
}

// Orthonormal axes with the unit vector n last.
__device__ __forceinline__ void frame_about(const double n[3], float ax[3][3])
{
    const double a[3] = {fabs(n[0]), fabs(n[1]), fabs(n[2])};
    const int k0 = a[0] <= a[1] && a[0] <= a[2] ? 0 : (a[1] <= a[2] ? 1 : 2);
    const double t[3] = {k0 == 0 ? 1.0 : 0.0, k0 == 1 ? 1.0 : 0.0, k0 == 2 ? 1.0 : 0.0};
    double u[3], v[3];
    ftd::cross3d(n, t, u);
    const double iu = 1.0 / sqrt(ftd::dot3d(u, u));
    for (int k = 0; k < 3; k++) u[k] *= iu;
    ftd::cross3d(n, u, v);
    for (int k = 0; k < 3; k++) {
        ax[0][k] = (float)u[k];
        ax[1][k] = (float)v[k];
        ax[2][k] = (float)n[k];
    }
}

// Half the surface of a box of half extents h: the smaller of two boxes about
// the same primitives is kept.
__device__ __forceinline__ float box_cost(const float h[3]) { return h[0] * h[1] + h[1] * h[2] + h[0] * h[2]; }

template <int W>
__device__ __forceinline__ float group_min(float v)
{
#pragma unroll
    for (int o = W / 2; o >= 1; o >>= 1) v = fminf(v, __shfl_xor(v, o));
    return v;
}
template <int W>
__device__ __forceinline__ float group_max(float v)
{
#pragma unroll
    for (int o = W / 2; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}
template <int W>
__device__ __forceinline__ double group_sum(double v)
{
#pragma unroll
    for (int o = W / 2; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Leaf boxes, kLeafLanes lanes per leaf: the smaller of the axis-aligned box
// of the vertices and one about an axis, for triangles the area-weighted mean
// normal, for crossing points the normal of their least-squares plane (three
// or more points that are not collinear).  A patch of a smooth surface is
// thin along that axis, so for a node far away the box's distance is close to
// the patch's.  naxis: that axis times its weight (area, or points), for the
// nodes above.  NaN vertices bound nothing (their distances never win).
constexpr int kLeafLanes = 16;
template <int MODE>
__global__ __launch_bounds__(kBS) void k_leaf_items(const uint64_t* sc, const uint32_t* first,
                                                    const uint32_t* leaf_bin, IndexGeom ig, const int32_t* pidx,
                                                    const float* ifp, const int4* tris, Item* items, float4* naxis)
{
    if (halted(sc)) return;
    const int64_t l = ((int64_t)blockIdx.x * kBS + threadIdx.x) / kLeafLanes;
    if (l >= cnt_leaves(sc)) return;                   // whole group
    constexpr int NV = MODE == 0 ? 1 : 3;
    const uint32_t sub = threadIdx.x % kLeafLanes, b = first[l], e = first[l + 1];
    auto verts = [&](uint32_t s, float v[3][3]) {
        const int32_t j = pidx[s];
        if (MODE == 0) {
            for (int k = 0; k < 3; k++) v[0][k] = ifp[3 * (int64_t)j + k];
        } else {
            tri_vertices(tris, ifp, j, v[0], v[1], v[2]);
        }
    };
    float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    double ns[3] = {0.0, 0.0, 0.0};                    // triangles: area vector; points: sum
    for (uint32_t s = b + sub; s < e; s += kLeafLanes) {
        float v[3][3];
        verts(s, v);
        for (int q = 0; q < NV; q++)
            for (int k = 0; k < 3; k++) {
                lo[k] = fminf(lo[k], v[q][k]);
                hi[k] = fmaxf(hi[k], v[q][k]);
            }
        if (MODE == 1) {
            double e0[3], e1[3], nn[3];
            for (int k = 0; k < 3; k++) { e0[k] = (double)v[1][k] - v[0][k]; e1[k] = (double)v[2][k] - v[0][k]; }
            ftd::cross3d(e0, e1, nn);
            for (int k = 0; k < 3; k++) ns[k] += nn[k];
        } else {
            for (int k = 0; k < 3; k++) ns[k] += v[0][k];
        }
    }
    float c[3], hb[3];
    for (int k = 0; k < 3; k++) {
        lo[k] = group_min<kLeafLanes>(lo[k]);
        hi[k] = group_max<kLeafLanes>(hi[k]);
        ns[k] = group_sum<kLeafLanes>(ns[k]);
        c[k] = 0.5f * (lo[k] + hi[k]);
        hb[k] = fmaxf(hi[k] - c[k], c[k] - lo[k]);
    }
    double n[3] = {0.0, 0.0, 0.0}, wt = 0.0;
    if (MODE == 1) {
        wt = sqrt(ftd::dot3d(ns, ns));
        if (wt > 0.0) for (int k = 0; k < 3; k++) n[k] = ns[k] / wt;
        else wt = 0.0;
    } else if (e - b >= 3) {
        double cov[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        const double cnt = (double)(e - b);
        for (uint32_t s = b + sub; s < e; s += kLeafLanes) {
            float v[3][3];
            verts(s, v);
            const double d0 = v[0][0] - ns[0] / cnt, d1 = v[0][1] - ns[1] / cnt, d2 = v[0][2] - ns[2] / cnt;
            cov[0] += d0 * d0; cov[1] += d1 * d1; cov[2] += d2 * d2;
            cov[3] += d0 * d1; cov[4] += d0 * d2; cov[5] += d1 * d2;
        }
        for (int k = 0; k < 6; k++) cov[k] = group_sum<kLeafLanes>(cov[k]);
        if (smallest_eigvec(cov, n)) wt = cnt;
    }
    float ax[3][3] = {{1.0f, 0.0f, 0.0f}, {0.0f, 1.0f, 0.0f}, {0.0f, 0.0f, 1.0f}};
    float h[3] = {hb[0], hb[1], hb[2]};
    double m[3] = {c[0], c[1], c[2]};
    if (wt > 0.0) {
        float fx[3][3];
        frame_about(n, fx);
        float l3[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, h3[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
        for (uint32_t s = b + sub; s < e; s += kLeafLanes) {
            float v[3][3];
            verts(s, v);
            for (int q = 0; q < NV; q++) {
                const float d0 = v[q][0] - c[0], d1 = v[q][1] - c[1], d2 = v[q][2] - c[2];
                for (int k = 0; k < 3; k++) {
                    const float t = __fmaf_rn(fx[k][2], d2, __fmaf_rn(fx[k][1], d1, fx[k][0] * d0));
                    l3[k] = fminf(l3[k], t);
                    h3[k] = fmaxf(h3[k], t);
                }
            }
        }
        float ho[3], mid[3];
        for (int k = 0; k < 3; k++) {
            l3[k] = group_min<kLeafLanes>(l3[k]);
            h3[k] = group_max<kLeafLanes>(h3[k]);
            mid[k] = 0.5f * (l3[k] + h3[k]);
            // the rounding of the projections: their terms are below 2 |hb|
            ho[k] = fmaxf(h3[k] - mid[k], mid[k] - l3[k]) + 0x1.0p-21f * (hb[0] + hb[1] + hb[2]);
        }
        if (box_cost(ho) < box_cost(hb)) {
            for (int k = 0; k < 3; k++) {
                h[k] = ho[k];
                for (int q = 0; q < 3; q++) {
                    ax[k][q] = fx[k][q];
                    m[q] += (double)mid[k] * fx[k][q];
                }
            }
        }
    }
    if (sub == 0) {
        items[l] = make_item(ig.grids[bin_field(ig, leaf_bin[l])], ax, m, h);
        naxis[l] = make_float4((float)(n[0] * wt), (float)(n[1] * wt), (float)(n[2] * wt), 0.0f);
    }
}

// Node boxes of one level, one wave per node with a child per lane: the
// smaller of two boxes that hold the children's, axis-aligned and about the
// weighted mean of their axes (signs aligned: two opposite sheets share
// theirs).  Everything in scaled coordinates.  Levels are fitted one after
// the other; nodes past the level's count leave at once.
__device__ __forceinline__ int64_t cnt_level(const uint64_t* lv, int level)
{
    const uint64_t v = level == 1 ? lv[0] >> 32 : level == 2 ? lv[1] : level == 3 ? lv[1] >> 32 : lv[2];
    return (int64_t)(v & 0xffffffffull);
}

__global__ __launch_bounds__(kBS) void k_node_items(const uint64_t* sc, int level, uint32_t off,
                                                    const uint32_t* first, Item* items, float4* naxis)
{
    if (halted(sc)) return;
    const int64_t n_nodes = cnt_leaves(sc) > 0 ? cnt_level(sc + S_LV, level) : 0;
    const int lane = ftd::lane_id();
    for (int64_t i = ((int64_t)blockIdx.x * kBS + threadIdx.x) >> 6; i < n_nodes; i += (int64_t)gridDim.x * (kBS / 64)) {
        const uint32_t g = off + (uint32_t)i, c0 = first[g], cnt = first[g + 1] - c0;
        const bool on = (uint32_t)lane < cnt;
        const Item it = items[c0 + (on ? lane : 0)];
        const float4 na = naxis[c0 + (on ? lane : 0)];
        const float4 r[3] = {row_values(it.x), row_values(it.y), row_values(it.z)};
        const float he[3] = {it.e.x, it.e.y, it.e.z};
        const bool open = __ballot(on && !(it.e.x <= 1e15f)) != 0ull;    // a child that admits every point
        float m[3];                                     // child centre: minus the rows' offsets along the axes
        for (int q = 0; q < 3; q++) {
            const float a0 = q == 0 ? r[0].x : q == 1 ? r[0].y : r[0].z, a1 = q == 0 ? r[1].x : q == 1 ? r[1].y : r[1].z,
                        a2 = q == 0 ? r[2].x : q == 1 ? r[2].y : r[2].z;
            m[q] = -__fmaf_rn(r[2].w, a2, __fmaf_rn(r[1].w, a1, r[0].w * a0));
        }
        const float r0x = __shfl(na.x, 0), r0y = __shfl(na.y, 0), r0z = __shfl(na.z, 0);
        const double sg = on ? (na.x * r0x + na.y * r0y + na.z * r0z < 0.0f ? -1.0 : 1.0) : 0.0;
        double ns[3] = {sg * na.x, sg * na.y, sg * na.z};
        for (int k = 0; k < 3; k++) ns[k] = group_sum<64>(ns[k]);
        const double wt = sqrt(ftd::dot3d(ns, ns));
        float fx[2][3][3] = {{{1.0f, 0.0f, 0.0f}, {0.0f, 1.0f, 0.0f}, {0.0f, 0.0f, 1.0f}}, {}};
        const bool axis = wt > 0.0;
        if (axis) {
            const double n[3] = {ns[0] / wt, ns[1] / wt, ns[2] / wt};
            frame_about(n, fx[1]);
        }
        float mid[2][3], h[2][3], far = 0.0f;
        for (int k = 0; k < 3; k++) far = fmaxf(far, group_max<64>(on ? fabsf(m[k]) : 0.0f));
        for (int t = 0; t < (axis ? 2 : 1); t++)
            for (int k = 0; k < 3; k++) {
                const float* a = fx[t][k];
                const float c = __fmaf_rn(a[2], m[2], __fmaf_rn(a[1], m[1], a[0] * m[0]));
                float rad = 0.0f;
                for (int q = 0; q < 3; q++)
                    rad += he[q] * fabsf(__fmaf_rn(a[2], r[q].z, __fmaf_rn(a[1], r[q].y, a[0] * r[q].x)));
                const float lo = group_min<64>(on ? c - rad : FLT_MAX), hi = group_max<64>(on ? c + rad : -FLT_MAX);
                mid[t][k] = 0.5f * (lo + hi);
                // centres, radii and projections are good to a few 2^-24 of the
                // farthest child centre's distance from the origin
                h[t][k] = fmaxf(hi - mid[t][k], mid[t][k] - lo) * (1.0f + 0x1.0p-20f) + 0x1.0p-19f * (far + 0.25f);
            }
        if (lane == 0) {
            const int t = axis && box_cost(h[1]) < box_cost(h[0]) ? 1 : 0;
            Item p;
            p.x = make_row(fx[t][0][0], fx[t][0][1], fx[t][0][2], -mid[t][0]);
            p.y = make_row(fx[t][1][0], fx[t][1][1], fx[t][1][2], -mid[t][1]);
            p.z = make_row(fx[t][2][0], fx[t][2][1], fx[t][2][2], -mid[t][2]);
            p.e = make_float4(h[t][0], h[t][1], h[t][2], 0.0f);
            items[g] = open || !(h[t][0] <= 1e15f && h[t][1] <= 1e15f && h[t][2] <= 1e15f) ? open_item() : p;
            naxis[g] = axis ? make_float4((float)ns[0], (float)ns[1], (float)ns[2], 0.0f) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    }
}

// ============================================================================
// Nearest-primitive search with the fused reinit epilogue
// ============================================================================
enum Epi : int { EPI_RAW = 0, EPI_INIT = 1, EPI_UPDATE = 2 };

struct QueryArgs {
    int64_t n_slots;                 // query slots (per-field Morton order, 64-padded)
    const float *sx, *sy, *sz;       // slot coordinates
    const int32_t* perm;             // slot -> node (-1: padding)
    const int32_t* tile_field;       // 64-slot tile -> field
    const int32_t* tile_list;        // launch order of the tiles, deep ones first (null: slot order)
    const uint64_t* n_deep;          // deep tiles at the head of tile_list (low 32 bits)
    const Grid* grids;               // per field: scaled coordinates
    const uint32_t* roots;           // field -> tree root (~0: no primitives)
    const uint32_t* first;           // children of each node, primitives of each leaf (LevelOff numbering)
    const Item* items;               // boxes of the same
    uint32_t leaf_end;               // indices below are leaves
    const float4* prec;              // point records (mode 0): coordinates, id
    const Item* titem;               // triangles' frames and rectangles (mode 1; null: from the records)
    const TriRec* trec;              // their records
    float band;                      // > 0: narrow band
    const float* ifp;
    const int4* tris;
    const double* phi_old;           // sign + retained values
    double* phi_out;
    double* phi_ifn;                 // nullable
    const uint64_t* retain;          // nullable
    int32_t* nearest;                // nullable
    int epi;
    double w_phi, w_ifn;
    uint32_t* clamped;               // narrow band: nodes clamped, per tile
    unsigned long long* stats;       // nullable: per distance bucket
    float h_est;                     // node spacing (statistics only)
    int probe;                       // a first candidate from the search for the tile's centre
    const uint64_t* sc;              // stage totals and halt flags
    uint32_t* queue;                 // counters, kQueueLine apart: deep tiles, then one per XCD
    ulonglong2* split_out;           // best and second key per lane of each part of a split tile (null: none split)
};

// The dispatcher hands workgroup b to XCD b % 8, each XCD with its own L2, so
// the tiles after the deep ones are dealt to the XCDs in runs of `chunk`
// consecutive ones (in Morton order, a compact region whose triangle and tree
// records its L2 keeps): the runs x, x + 8, x + 16, ... to XCD x.  At least 8
// runs each, that costly regions spread over all of them (one run each was
// slower), and up to 1024 tiles long (256^3; 512 is 1 % slower, 2048 0.5 %).
constexpr unsigned kXcds = 8;
struct XcdShare {
    uint32_t n, chunk, span;         // tiles in all, per run, per run of every XCD
    __device__ explicit XcdShare(uint32_t tiles) : n(tiles)
    {
        const uint32_t c = tiles / (kXcds * 8);
        chunk = c < 1u ? 1u : c > 1024u ? 1024u : c;
        span = kXcds * chunk;
    }
    __device__ uint32_t tiles(uint32_t x) const       // of XCD x
    {
        const uint32_t whole = n / span, rest = n - whole * span, at = x * chunk;
        return whole * chunk + (rest <= at ? 0u : rest - at < chunk ? rest - at : chunk);
    }
    __device__ uint32_t tile(uint32_t x, uint32_t k) const   // the k-th of XCD x
    {
        return k / chunk * span + x * chunk + k % chunk;
    }
};

// Margin of the box prune: a box is skipped only if its lower bound exceeds
// the best distance by more than the float rounding of both (relative) plus
// an absolute floor for near-zero distances.
__device__ __forceinline__ float prune_bound(float best2)
{
    return __fmaf_rn(best2, 1.0f + 0x1.0p-16f, 1.0e-30f);
}

// A candidate as one 64-bit key: the distance's bits above the primitive's
// id.  Distances are non-negative, so their bit patterns order as their
// values, and key order is the order (distance, then lower id); no candidate
// is id -1, the largest id as unsigned.
__device__ __forceinline__ uint64_t cand_key(float d, int32_t j)
{
    return ((uint64_t)__float_as_uint(d) << 32) | (uint32_t)j;
}

// End of a node's search.  Points: the nearest (distance, lowest id).
// Triangles: the best two by FP32 squared distance, for the FP64 settle.
struct Found {
    float x, y, z;
    uint64_t bkey, skey;
    __device__ __forceinline__ float best() const { return __uint_as_float((uint32_t)(bkey >> 32)); }
    __device__ __forceinline__ int32_t bj() const { return (int32_t)(uint32_t)bkey; }
    __device__ __forceinline__ float sec() const { return __uint_as_float((uint32_t)(skey >> 32)); }
    __device__ __forceinline__ int32_t sj() const { return (int32_t)(uint32_t)skey; }
};

// Epilogue of one node (EuclideanDistance.cu:54-57, LevelSet.cpp:438-448, 74,
// 148): sign from phi_old < 0, retained value at crossing-edge nodes, blend.
__device__ __forceinline__ void node_epilogue(const QueryArgs& a, int64_t node, double d, int32_t near)
{
    const double po = a.phi_old[node];
    const double dn = (po < 0.0) ? -d : d;
    if (a.phi_ifn) a.phi_ifn[node] = dn;
    if (a.nearest) a.nearest[node] = near;
    double out = dn;
    if (a.epi == EPI_UPDATE) {
        const double kept = (a.retain && ftd::get_bit(a.retain, node)) ? po : dn;
        out = a.w_phi * kept + a.w_ifn * dn;
    }
    a.phi_out[node] = out;
}

// FP64 squared distance from point (x, y, z) to triangle f of the interface.
__device__ inline double node_tri_dist2(const QueryArgs& a, float x, float y, float z, int32_t f)
{
    const int4 t = a.tris[f];
    const float p[3] = {x, y, z};
    float va[3], vb[3], vc[3];
    for (int k = 0; k < 3; k++) {
        va[k] = a.ifp[3 * (int64_t)t.x + k];
        vb[k] = a.ifp[3 * (int64_t)t.y + k];
        vc[k] = a.ifp[3 * (int64_t)t.z + k];
    }
    return ftd::tri_dist2_f64(p, va, vb, vc);
}

// End of the search of one node, then its epilogue.  Points: the float
// distance, as the reference.  Triangles: the FP32 search knows the nearest
// triangle up to its rounding (at 256^3 float rounding alone nears 1e-5 h),
// so the best and, when that close, the runner-up are evaluated in FP64; the
// lower wins, ties to the lower id.  No candidate: +-band in a narrow band,
// else +-FLT_MAX.
template <int MODE>
__device__ __forceinline__ void finish_node(const QueryArgs& a, const Found& S, int64_t node)
{
    if (MODE == 0) {
        const float d = (a.band > 0.0f && S.bj() < 0) ? a.band : S.best();
        node_epilogue(a, node, (double)d, S.bj());
    } else {
        double d;
        int32_t near = S.bj();
        if (near >= 0) {
            double d2 = node_tri_dist2(a, S.x, S.y, S.z, near);
            const int32_t sj = S.sj();
            const bool close = sj >= 0 && S.sec() <= S.best() * (1.0f + 0x1.0p-16f);
            if (close) {
                const double e2 = node_tri_dist2(a, S.x, S.y, S.z, sj);
                if (e2 < d2 || (e2 == d2 && sj < near)) { d2 = e2; near = sj; }
            }
            d = sqrt(d2);
        } else {
            d = (double)(a.band > 0.0f ? a.band : FLT_MAX);
        }
        node_epilogue(a, node, d, near);
    }
}

// Query schedule.  A tile deep inside a closed surface is the longest: near
// the middle every triangle is nearly equidistant, and the exact search must
// certify them all.  Its time grows with the square of the depth (256^3, 64
// spheres: 3.3 ms at phi_old = -29 h where the mean tile takes 0.14 ms), so
// such tiles, started late or in a small field, set the kernel's end.  A tile
// is deep when one of its nodes has phi_old <= -kDeepTile split_h h of its
// field: the deep tiles are listed first and are what the waves start with; the
// rest keep their slot (Morton) order.  A tile is very deep from -split_h h: it is searched by
// kSplitParts waves, each with all 64 nodes but testing only the leaves l with
// l % kSplitParts equal to its part, and k_split_merge combines the parts.
// Each part repeats the walk above the leaves, so splitting costs work, and
// the depth from which it pays goes down with the launch's own length: split_h
// = 25 for 2^18 tiles (256^3 nodes), as the square root of the tiles below
// that, at least 2.5 (a 32^3 sphere: 127 -> 69 us; at 256^3 15 h in place of
// 25 h is 1% slower, 8 parts in place of 4 the same).  At most split_tiles_cap
// tiles per launch are split (the parts' results take kSplitParts x 1 KiB per
// tile); the rest run whole.  The split only changes which wave tests a leaf:
// each node's result is the same.
constexpr float kDeepTile = 0.4f;            // of split_tile_h
constexpr float kSplitTileH = 25.0f;
constexpr float kSplitTileMinH = 2.5f;
inline float split_tile_h(int64_t n_tiles)
{
    const float h = kSplitTileH * std::sqrt((float)n_tiles / 262144.0f);
    return std::min(kSplitTileH, std::max(kSplitTileMinH, h));
}
constexpr int kSplitParts = 4;
constexpr int64_t kSplitCap = 1024;

__host__ __device__ inline int64_t split_tiles_cap(int64_t n_tiles)
{
    const int64_t cap = n_tiles / 64 > kSplitCap ? n_tiles / 64 : kSplitCap;
    return n_tiles < cap ? n_tiles : cap;
}

// One wave per tile: cls[t] = 2 when some node of tile t is very deep, 1 when
// deep, else 0.
__global__ __launch_bounds__(kBS) void k_tile_deep(int64_t n_tiles, const int32_t* perm, const double* phi,
                                                   const int32_t* tile_field, const Grid* grids, float deep_h,
                                                   float split_h, uint32_t* cls, const uint64_t* sc)
{
    if (halted(sc)) return;
    const int64_t t = ((int64_t)blockIdx.x * kBS + threadIdx.x) >> 6;
    if (t >= n_tiles) return;                          // whole wave
    const int32_t node = perm[t * 64 + ftd::lane_id()];
    const float h = grids[tile_field[t]].h;
    const double p = node >= 0 ? phi[node] : 0.0;
    const uint64_t m1 = __ballot(p <= -(double)(deep_h * h));
    const uint64_t m2 = __ballot(p <= -(double)(split_h * h));
    if (ftd::lane_id() == 0) cls[t] = m2 ? 2u : (m1 ? 1u : 0u);
}

// Stable partition from the exclusive scan ex of LoadTileClass(cls) (K deep
// tiles, K2 of them very deep): the very deep tiles to list[0, K2), the other
// deep ones to list[K2, K), the rest after them, each in tile order.
__global__ __launch_bounds__(kBS) void k_tile_list(int64_t n_tiles, const uint32_t* cls, const uint64_t* ex,
                                                   const uint64_t* sc, int32_t* list)
{
    if (halted(sc)) return;
    const int64_t t = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (t >= n_tiles) return;
    const uint64_t tot = sc[S_DEEP];
    const int64_t K = (int64_t)(uint32_t)tot, K2 = (int64_t)(tot >> 32);
    const int64_t e1 = (int64_t)(uint32_t)ex[t], e2 = (int64_t)(ex[t] >> 32);
    const uint32_t c = cls[t];
    const int64_t at = c == 2 ? e2 : (c == 1 ? K2 + (e1 - e2) : K + (t - e1));
    list[at] = (int32_t)t;
}

// ---- the search of one tile -------------------------------------------------
// Traversal counts of a tile (FT_QUERY_STATS).
struct TileStats {
    uint32_t nodes = 0, boxes = 0, leaves = 0, prims = 0, pairs = 0;
};

template <int MODE>
__device__ __forceinline__ void record_stats(const QueryArgs& a, const Found& S, int64_t node, const TileStats& t)
{
    // buckets: distance < 2h, < 8h, < 32h, beyond; +4 when phi < 0
    const float dd = MODE == 0 ? S.best() : sqrtf(S.best());
    const float hh = a.h_est;
    int bkt = dd < 2 * hh ? 0 : dd < 8 * hh ? 1 : dd < 32 * hh ? 2 : 3;
    if (a.phi_old[node] < 0.0) bkt += 4;
    unsigned long long* st = a.stats + 6 * bkt;
    atomicAdd(&st[0], 1ull);
    atomicAdd(&st[1], (unsigned long long)t.nodes);
    atomicAdd(&st[2], (unsigned long long)t.boxes);
    atomicAdd(&st[3], (unsigned long long)t.leaves);
    atomicAdd(&st[4], (unsigned long long)t.prims);
    atomicAdd(&st[5], (unsigned long long)t.pairs);
}

typedef float v4f __attribute__((ext_vector_type(4)));

// Squared length with the parts' negative values as 0 and each part at most
// 1 (scaled coordinates: the clamp is the subtraction's own output modifier,
// one instruction; a part cut to 1 only lowers the bound).
__device__ __forceinline__ float sat(float v) { return __builtin_amdgcn_fmed3f(v, 0.0f, 1.0f); }
__device__ __forceinline__ float box_d2(float x, float y, float z, const float4& e)
{
    const float dx = sat(fabsf(x) - e.x), dy = sat(fabsf(y) - e.y), dz = sat(fabsf(z) - e.z);
    return __fmaf_rn(dx, dx, __fmaf_rn(dy, dy, dz * dz));
}
// The same to a triangle's rectangle (no extent along its normal).
__device__ __forceinline__ float rect_d2(float x, float y, float z, const float2& e)
{
    const float dx = sat(fabsf(x) - e.x), dy = sat(fabsf(y) - e.y);
    return __fmaf_rn(dx, dx, __fmaf_rn(dy, dy, z * z));
}

// Least of the wave's keys (the lanes of a wave run together; every lane
// holds one): row shifts, then broadcasts over the rows, the total in lane 63.
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v)
{
#define FT_DPP_MIN(ctrl) \
    v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)0xffffffffu, (int)v, ctrl, 0xf, 0xf, false))
    FT_DPP_MIN(0x111);                        // row_shr 1, 2, 4, 8
    FT_DPP_MIN(0x112);
    FT_DPP_MIN(0x114);
    FT_DPP_MIN(0x118);
    FT_DPP_MIN(0x142);                        // row_bcast 15, 31
    FT_DPP_MIN(0x143);
#undef FT_DPP_MIN
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// LDS of one wave.  The nodes' keys, coordinates and pruning bounds are kept
// here and not in registers, because the search works on (node, primitive)
// pairs, whose node is any lane's.
constexpr int kQueue = 64 + 256;              // pairs: less than a wave's, then one group's
template <int MODE>
struct __align__(16) WaveLds {
    unsigned long long best[64];
    unsigned long long sec[MODE == 1 ? 64 : 1];
    float px[64], py[64], pz[64];
    uint2 queue[kQueue];                      // (primitive slot, node's lane); the seed search's lists before
    float thr[MODE == 0 ? 128 : 64];
    uint32_t range[kLevels - 1][66];          // per level of the walk: the children's ranges (first[])
    uint4 stack[kLevels - 1];                 // lists of the levels above: first child, mask
};

// Orders the wave's LDS stores before its loads (a wave runs its lanes
// together: a wave-scope fence waits for its own LDS accesses).
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Search of the tile of 64 nodes held by a wave, one node per lane.
//
// Pruning is separated from the exact distances:
//  - four boxes (the children of a node, or the rectangles of a leaf's
//    triangles) are taken against the 64 nodes by four 16 x 16 x 16 matrix
//    instructions on halves (Item): the coordinates of 16 nodes along the 12 box
//    axes at once.
//    In the product lane l holds box l / 16 and node l % 16 of the 16, its
//    three coordinates in three registers, so the distance to the box is 6 or
//    7 instructions for 64 (node, box) pairs and a compare against the node's
//    bound.  Crossing points take 16 per FP32 instruction (16 x 16 x 4):
//    |q|^2 - 2 p.q about the tile's centre against the bound less |p|^2.
//  - the pairs that pass go to a queue in LDS, and every 64 of them are
//    evaluated together, one pair per lane, whichever nodes and primitives
//    they are: a primitive that concerns 9 nodes costs 9 lanes and not 64.
//    Their keys go to the nodes' best (and second) by LDS minimum.
//  - nothing is sorted: a first search for the tile's centre alone (children
//    on the lanes, nearest first) finds a primitive near every node's nearest
//    before the walk, and with bounds that good the order of the walk is
//    worth 4% (in a model of the traversal at 256^3; without that first
//    search the walk takes twice the boxes and triangles).
//  - RECORDS: the triangles' rectangles are formed from their records where
//    they are read, instead of from items of their own (64 bytes a triangle):
//    for an allocation-free call whose scratch cannot take both.
// Every cut is a lower bound compared with the node's best so far raised by
// its rounding: scaled coordinates are good to 2^-20 along each axis, so the
// bound is (sqrt(best) + 2^-19)^2; results are the exact search's.
//
// What bounds it: vector issue (76-80% of its rate at 256^3: 12.0k vector
// instructions per tile).  256^3, 64 spheres, full
// domain: 5.9-6.3 ms, against 9.1-9.5 ms for a wave-wide walk of a binary tree that
// tested every box and triangle on all 64 lanes (19.9k instructions per tile);
// crossing points 3.2 against 3.9 ms.
template <int MODE, bool STATS, bool RECORDS = false>
struct TileSearch {
    const QueryArgs& a;
    WaveLds<MODE>& lds;
    const int lane;
    uint32_t qn = 0;                          // queued pairs
    float thr[4];                             // scaled bounds of nodes 16 cb + lane % 16
    v4h B[4];                                 // matrix operand of those nodes: coordinates and 1, split (see Item)
    float inv_s;
    float cen[3], pp = 0.0f;                  // tile centre; points: |p - cen|^2 of the lane's node, lowered
    float rel[MODE == 0 ? 4 : 1];             // points: operand about the centre
    float org[RECORDS ? 3 : 1];               // origin of the scaled coordinates
    TileStats st;

    __device__ __forceinline__ TileSearch(const QueryArgs& q, WaveLds<MODE>& l, int ln) : a(q), lds(l), lane(ln) {}

    // The lane as a value the compiler takes for new: what is derived from it
    // is formed again here rather than kept (or spilled) across the search.
    __device__ __forceinline__ int fresh_lane() const
    {
        int l = lane;
        asm volatile("" : "+v"(l));
        return l;
    }

    __device__ __forceinline__ float node_best(int i) const
    {
        return __uint_as_float((uint32_t)(lds.best[i] >> 32));
    }

    // The nodes' bounds from their keys.
    __device__ __forceinline__ void refresh()
    {
        wave_lds_sync();
        const float b = node_best(lane);
        const float bnd = prune_bound(MODE == 0 ? b * b : b);
        const float s = __fmaf_rn(ftd::sqrt_lb(bnd) * inv_s, 1.0f + 0x1.0p-20f, 0x1.0p-19f);
        lds.thr[lane] = s * s;
        if (MODE == 0) lds.thr[64 + lane] = __fmaf_rn(bnd, 1.0f + 0x1.0p-18f, -pp);
        wave_lds_sync();
#pragma unroll
        for (int cb = 0; cb < 4; cb++) thr[cb] = lds.thr[16 * cb + (lane & 15)];
    }

    // The exact FP32 distance of the queue's last n (<= 64) pairs.
    __device__ __forceinline__ void flush(uint32_t n)
    {
        wave_lds_sync();
        const bool on = (uint32_t)lane < n;
        const uint2 p = lds.queue[qn - n + (on ? lane : 0)];
        qn -= n;
        if (STATS) st.pairs += n;
        const float x = lds.px[p.y], y = lds.py[p.y], z = lds.pz[p.y];
        if (MODE == 0) {
            const float4 r = a.prec[p.x];
            const float dx = r.x - x, dy = r.y - y, dz = r.z - z;
            const float d = sqrtf(dx * dx + dy * dy + dz * dz);        // EuclideanDistance.cu:20-28
            if (on) atomicMin(&lds.best[p.y], (unsigned long long)cand_key(d, __float_as_int(r.w)));
        } else {
            const TriRec r = a.trec[p.x];
            const uint64_t key = cand_key(ftd::tri_dist2(x, y, z, r), ftd::tri_id(r));
            if (on) {
                // a key that is beaten, or beats one, leaves the loser to the second
                const uint64_t old = atomicMin(&lds.best[p.y], (unsigned long long)key);
                if (old != key) atomicMin(&lds.sec[p.y], (unsigned long long)(old > key ? old : key));
            }
        }
        refresh();
    }

    // Queues the (slot, node) pairs of the lanes in m.
    __device__ __forceinline__ void enqueue(uint64_t m, uint32_t slot, uint32_t node)
    {
        const uint32_t at = qn + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        if (__builtin_amdgcn_inverse_ballot_w64(m)) lds.queue[at] = make_uint2(slot, node);
        qn += (uint32_t)__popcll(m);
    }

    // Boxes it[0..3] of the n (1..4, more count as 4) left against the nodes:
    // passing (box, node) pairs per 16 nodes.
    __device__ __forceinline__ static float item_d2(const v4f& p, const float4& e) { return box_d2(p[0], p[1], p[2], e); }
    __device__ __forceinline__ static float item_d2(const v4f& p, const float2& e) { return rect_d2(p[0], p[1], p[2], e); }
    template <class E>
    __device__ __forceinline__ void cull4(v4h av, const E& e, uint32_t n, uint64_t m[4]) const
    {
        const uint64_t live = n >= 4 ? ~0ull : (1ull << (16 * n)) - 1ull;
        v4f d[4];
#pragma unroll
        for (int cb = 0; cb < 4; cb++) d[cb] = __builtin_amdgcn_mfma_f32_16x16x16f16(av, B[cb], v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
        for (int cb = 0; cb < 4; cb++) m[cb] = __ballot(item_d2(d[cb], e) <= thr[cb]) & live;
    }
    // This lane's element of the matrix operand of items it[0..3], and the
    // extents of item lane / 16.  (Up to three items past the last are read.)
    template <class E>
    __device__ __forceinline__ static void load4(const Item* it, int lane, v4h& av, E& e)
    {
        const v4h* f = reinterpret_cast<const v4h*>(it);       // 8 per item: a row's hi and lo in turn
        av = f[(uint32_t)(((lane & 15) >> 2) * 8 + (lane & 3) * 2 + (lane >> 5))];
        e = *reinterpret_cast<const E*>(f + (uint32_t)((lane >> 4) * 8 + 6));
    }

    // The same of the triangles in slots s to s + 3, of which `left` are the
    // leaf's (the rest as its last).  A rectangle's offsets formed in FP32 are
    // good to 2^-22 of a scaled unit, beside the product's 2^-22.8, of the 2^-20
    // that the bounds allow.
    __device__ __forceinline__ void load_tris(uint32_t s, uint32_t left, int lane, v4h& av, float2& e) const
    {
        if (!RECORDS) {
            load4(a.titem + s, lane, av, e);
            return;
        }
        const float4* r = reinterpret_cast<const float4*>(a.trec + s);          // 5 per record: a, u, v, n, i
        auto record = [&](int k) { return r + 5u * ((uint32_t)k < left ? (uint32_t)k : left - 1u); };
        const float4* t = record((lane & 15) >> 2);
        const int j = lane & 3;                                // row u, v or n (the fourth is a spare one)
        const float4 o = t[0], x = t[j < 2 ? 1 + j : 3];
        const float half = j == 0 ? 0.5f * x.w : j == 1 ? 0.5f * t[3].w : 0.0f;
        const float dx = o.x - org[0], dy = o.y - org[1], dz = o.z - org[2];
        const float w = -(__fmaf_rn(dz, x.z, __fmaf_rn(dy, x.y, dx * x.x)) + half) * inv_s;
        const Row row = make_row(x.x, x.y, x.z, w);
        av = lane < 32 ? row.hi : row.lo;
        const float4* b = record(lane >> 4);
        const float up = 0.5f * inv_s * (1.0f + 0x1.0p-20f);
        e = make_float2(b[1].w * up, b[3].w * up);
    }

    // Which of the children [c0, c0 + cnt), cnt <= 64, some node admits; their
    // ranges go to lds.range[d].
    __device__ __forceinline__ uint64_t admitted(uint32_t c0, uint32_t cnt, int d)
    {
        const int lane = fresh_lane();
        v4h av;
        float4 e;
        load4(a.items + c0, lane, av, e);
        const uint32_t f = a.first[c0 + lane], fe = a.first[c0 + cnt];   // (past the children: unused)
        if (STATS) {
            st.nodes++;
            st.boxes += cnt;
        }
        uint32_t keep = 0;                             // lane k: child k's nodes (any of the 4 sets of 16)
        for (uint32_t i = 0; i < cnt; i += 4) {
            v4h av1 = av;
            float4 e1 = e;
            if (i + 4 < cnt) load4(a.items + c0 + i + 4, lane, av1, e1);
            uint64_t m[4];
            cull4(av, e, cnt - i, m);
            const uint64_t u = (m[0] | m[1]) | (m[2] | m[3]);
            const uint32_t mine = (uint32_t)(u >> (16 * (lane & 3))) & 0xffffu;
            keep = (uint32_t)lane >> 2 == i >> 2 ? mine : keep;
            av = av1;
            e = e1;
        }
        lds.range[d][lane] = f;
        lds.range[d][cnt] = fe;                        // (after the lanes' own: a wave's LDS writes keep their order)
        wave_lds_sync();
        return __ballot(keep != 0u);
    }

    // The points that reach any of the boxes [c0, c0 + cnt), cnt <= 64, which
    // then admit nothing more.
    __device__ __forceinline__ uint64_t reached(uint32_t c0, uint32_t cnt)
    {
        const int lane = fresh_lane();
        uint64_t all[4] = {0, 0, 0, 0};
        v4h av;
        float4 e;
        load4(a.items + c0, lane, av, e);
        for (uint32_t i = 0; i < cnt; i += 4) {
            v4h av1 = av;
            float4 e1 = e;
            if (i + 4 < cnt) load4(a.items + c0 + i + 4, lane, av1, e1);
            uint64_t m[4];
            cull4(av, e, cnt - i, m);
#pragma unroll
            for (int cb = 0; cb < 4; cb++) all[cb] |= m[cb];
            av = av1;
            e = e1;
        }
        uint64_t hit = 0;
#pragma unroll
        for (int cb = 0; cb < 4; cb++) {
            uint64_t v = all[cb] | (all[cb] >> 32);
            v = (v | (v >> 16)) & 0xffffull;
            hit |= v << (16 * cb);
            if ((v >> (lane & 15)) & 1ull) thr[cb] = -1.0f;
        }
        return hit;
    }

    // Range of element b of list d.
    __device__ __forceinline__ void range_of(int d, uint32_t b, uint32_t& s0, uint32_t& s1) const
    {
        s0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds.range[d][b]);
        s1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds.range[d][b + 1]);
    }

    // The next leaf of a list: the first element of mask, taken out of it.
    // False when there is none.
    __device__ __forceinline__ bool next_leaf(uint64_t& mask, int d, uint32_t& s0, uint32_t& s1)
    {
        if (!mask) return false;
        const uint32_t b = (uint32_t)(__ffsll((unsigned long long)mask) - 1);
        mask &= mask - 1;
        range_of(d, b, s0, s1);
        if (STATS) {
            st.leaves++;
            st.prims += s1 - s0;
        }
        return true;
    }

    // The primitives of the leaves of mask (list d), the next group's loads in
    // flight while one is taken, across leaves.
    __device__ __forceinline__ void leaves(uint64_t mask, int d)
    {
        const int lane = fresh_lane();
        uint32_t s, s1;
        if (!next_leaf(mask, d, s, s1)) return;
        if (MODE == 1) {
            v4h av;
            float2 e;
            load_tris(s, s1 - s, lane, av, e);
            for (;;) {
                uint32_t ns = s + 4, ns1 = s1;
                const bool more = ns < s1 || next_leaf(mask, d, ns, ns1);
                v4h av1 = av;
                float2 e1 = e;
                if (more) load_tris(ns, ns1 - ns, lane, av1, e1);
                uint64_t m[4];
                cull4(av, e, s1 - s, m);
                if ((m[0] | m[1]) | (m[2] | m[3])) {
#pragma unroll
                    for (int cb = 0; cb < 4; cb++)
                        if (m[cb]) enqueue(m[cb], s + (uint32_t)(lane >> 4), (uint32_t)(16 * cb + (lane & 15)));
                    while (qn >= 64) flush(64);
                }
                if (!more) return;
                av = av1;
                e = e1;
                s = ns;
                s1 = ns1;
            }
        } else {
            const int k = lane >> 4;
            const uint32_t i = (uint32_t)(lane & 15);
            float4 r = a.prec[s + (i < s1 - s ? i : 0u)];
            for (;;) {
                uint32_t ns = s + 16, ns1 = s1;
                const bool more = ns < s1 || next_leaf(mask, d, ns, ns1);
                const float qx = r.x - cen[0], qy = r.y - cen[1], qz = r.z - cen[2];
                if (more) r = a.prec[ns + (i < ns1 - ns ? i : 0u)];
                const float qq = __fmaf_rn(qz, qz, __fmaf_rn(qy, qy, qx * qx)) * (1.0f - 0x1.0p-18f);
                const float q3 = k == 0 ? qx : k == 1 ? qy : qz;
                const float av = k == 3 ? qq : -2.0f * q3;
                v4f p[4];
#pragma unroll
                for (int cb = 0; cb < 4; cb++)
                    p[cb] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, rel[cb], v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                const uint32_t left = s1 - s;
#pragma unroll
                for (int q = 0; q < 4; q++) {              // points 4 (lane / 16) + q of the 16
                    const uint32_t pi = (uint32_t)(4 * k + q);
                    const uint64_t live = __ballot(pi < left);
                    uint64_t m[4];
#pragma unroll
                    for (int cb = 0; cb < 4; cb++)
                        m[cb] = __ballot(p[cb][q] <= lds.thr[64 + 16 * cb + (int)i]) & live;
                    if ((m[0] | m[1]) | (m[2] | m[3])) {
#pragma unroll
                        for (int cb = 0; cb < 4; cb++)
                            if (m[cb]) enqueue(m[cb], s + pi, 16 * cb + i);
                        while (qn >= 64) flush(64);
                    }
                }
                if (!more) return;
                s = ns;
                s1 = ns1;
            }
        }
    }

    // Squared distance, scaled, of a scaled point to an item's box, from the
    // rows' upper halves alone (2^-12 of a unit: a seed need not be exact).
    __device__ __forceinline__ static float box_of(const Item& it, float x, float y, float z)
    {
        auto at = [&](const Row& r) {
            return __fmaf_rn((float)r.hi[0], x, __fmaf_rn((float)r.hi[1], y, __fmaf_rn((float)r.hi[2], z, (float)r.hi[3])));
        };
        return box_d2(at(it.x), at(it.y), at(it.z), it.e);
    }

    // The node just above the leaves with the leaf box nearest to the point
    // (x, y, z) (scaled), and a primitive of that leaf near it: the children of
    // a node one per lane, nearest first, boxes beyond the nearest leaf so far
    // left out, as are those beyond `best` (squared, scaled).  At most
    // kSeedSteps steps (the centre of a sphere would visit all of it): any
    // primitive will do.
    static constexpr int kSeedSteps = 48;
    __device__ __forceinline__ void seed(uint32_t root, float x, float y, float z, float best, uint32_t& slot, uint32_t& node)
    {
        // per level, 64 each: the children's bounds, and their ranges
        float* lists = reinterpret_cast<float*>(lds.queue);
        uint32_t* begins = reinterpret_cast<uint32_t*>(lds.queue) + 64 * (kLevels - 2);
        uint32_t f0, fb, fe, cur = root, s0 = 0, s1 = 0;
        float lb;
        int d = 0;
        auto enter = [&](uint32_t c0, uint32_t c1) {   // the children [c0, c1)
            f0 = c0;
            fb = a.first[c0 + lane];
            fe = a.first[c0 + lane + 1];
            lb = (uint32_t)lane < c1 - c0 ? box_of(a.items[c0 + lane], x, y, z) : INFINITY;
        };
        enter(ftd::cload(a.first, root), ftd::cload(a.first, root + 1));
        for (int step = 0; step < kSeedSteps; step++) {
            const uint32_t key = wave_min_u32((__float_as_uint(lb) & ~63u) | (uint32_t)lane);
            const uint32_t sel = key & 63u;
            const bool nearer = __uint_as_float(key & ~63u) < best;
            const uint32_t g0 = (uint32_t)__builtin_amdgcn_readlane((int)fb, sel), g1 = (uint32_t)__builtin_amdgcn_readlane((int)fe, sel);
            const bool above = f0 >= a.leaf_end;       // the children are nodes
            if (nearer && above) {
                if ((uint32_t)lane == sel) lb = INFINITY;
                lists[64 * d + lane] = lb;
                begins[128 * d + lane] = fb;
                begins[128 * d + 64 + lane] = fe;
                if (lane == 0) lds.stack[d].x = f0;
                d++;
                cur = f0 + sel;
                enter(g0, g1);
                continue;
            }
            if (nearer) {
                best = __uint_as_float(key & ~63u);
                s0 = g0;
                s1 = g1;
                node = cur;
            }
            if (d == 0) break;
            d--;
            wave_lds_sync();
            lb = lists[64 * d + lane];
            fb = begins[128 * d + lane];
            fe = begins[128 * d + 64 + lane];
            f0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds.stack[d].x);
        }
        wave_lds_sync();
        if (s0 == s1) return;
        // a lane past the leaf loses to any of its primitives, also to one whose
        // distance is not a number (its bits are above infinity's)
        uint32_t key = ~0u;
        if (s0 + lane < s1) {
            float t;
            if (RECORDS) {
                t = ftd::tri_dist2(cen[0], cen[1], cen[2], a.trec[s0 + lane]);
            } else if (MODE == 1) {
                t = box_of(a.titem[s0 + lane], x, y, z);
            } else {
                const float4 r = a.prec[s0 + lane];
                const float dx = (r.x - cen[0]) * inv_s, dy = (r.y - cen[1]) * inv_s, dz = (r.z - cen[2]) * inv_s;
                t = __fmaf_rn(dx, dx, __fmaf_rn(dy, dy, dz * dz));
            }
            const uint32_t inf = 0x7f800000u, u = __float_as_uint(t);
            key = ((u < inf ? u : inf) & ~63u) | (uint32_t)lane;
        }
        slot = s0 + (wave_min_u32(key) & 63u);
    }

    // The leaves of node g; part of parts: only leaves l % parts == part.
    __device__ __forceinline__ uint64_t of_part(uint64_t mask, uint32_t c0, int parts, int part) const
    {
        if (parts == 1) return mask;
        return __ballot(((mask >> lane) & 1ull) && (int)((c0 + (uint32_t)lane) % (uint32_t)parts) == part);
    }

    // Walks the tree at root: first the node `start` above the leaves (~0:
    // none), whose primitives bring most nodes near their final bound, then
    // the rest.
    __device__ __forceinline__ void walk(uint32_t root, uint32_t start, int parts, int part)
    {
        bool first = start != ~0u && start != root;
        const uint32_t skip = first ? start : ~0u;
        uint32_t c0 = ftd::cload(a.first, first ? start : root), c1 = ftd::cload(a.first, (first ? start : root) + 1);
        int sp = 0;                                    // list sp: the children of a node
        for (;;) {
            uint32_t f0 = c0;                          // the list's first child, and those still to visit
            uint64_t mask = admitted(c0, c1 - c0, sp);
            if (f0 < a.leaf_end) {
                leaves(of_part(mask, f0, parts, part), sp);
                mask = 0;
            }
            if (first) {
                first = false;
                c0 = ftd::cload(a.first, root);
                c1 = ftd::cload(a.first, root + 1);
                continue;
            }
            uint32_t b;
            do {
                while (!mask) {                        // back to a list with something left
                    if (sp == 0) {
                        if (qn) flush(qn);
                        return;
                    }
                    sp--;
                    const uint4 t = lds.stack[sp];
                    f0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)t.x);
                    mask = (uint32_t)__builtin_amdgcn_readfirstlane((int)t.y) |
                           ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)t.z) << 32);
                }
                b = (uint32_t)(__ffsll((unsigned long long)mask) - 1);
                mask &= mask - 1;
            } while (f0 + b == skip);
            range_of(sp, b, c0, c1);
            if (lane == 0) lds.stack[sp] = make_uint4(f0, (uint32_t)mask, (uint32_t)(mask >> 32), 0u);
            sp++;                                      // at most kLevels - 2: a leaf is no list
        }
    }
};

// The key of a node without a candidate.
template <int MODE>
__device__ __forceinline__ uint64_t no_key(const QueryArgs& a)
{
    return MODE == 0 ? cand_key(a.band > 0.0f ? a.band : FLT_MAX, -1)
                     : cand_key(a.band > 0.0f ? a.band * a.band : INFINITY, -1);
}

// A wave's tile: 64 consecutive slots of one field in Morton order.
// split >= 0: part split % kSplitParts of split tile split / kSplitParts,
// whose best and second keys go to a.split_out instead of the epilogue.
template <int MODE, bool STATS, bool RECORDS>
__device__ __forceinline__ void search_tile(const QueryArgs& a, int64_t base, WaveLds<MODE>& lds, int split = -1)
{
    // opaque to the compiler, which would else hoist everything that depends on
    // the lane alone out of the work queue's loop, and spill it
    int lane = ftd::lane_id();
    asm volatile("" : "+v"(lane));
    TileSearch<MODE, STATS, RECORDS> S(a, lds, lane);
    const int64_t slot = base + lane;
    const int32_t node = a.perm[slot];                 // -1: padding lane
    Found F;
    F.x = a.sx[slot]; F.y = a.sy[slot]; F.z = a.sz[slot];
    const int field = __builtin_amdgcn_readfirstlane(a.tile_field[base >> 6]);
    const uint32_t root = (uint32_t)__builtin_amdgcn_readfirstlane((int)ftd::cload(a.roots, field));
    const uint64_t none = no_key<MODE>(a);
    F.bkey = F.skey = none;
    if (root != ~0u) {                                 // the field has primitives
        const Grid* g = a.grids + field;
        const float ox = ftd::cload(&g->org[0], 0), oy = ftd::cload(&g->org[1], 0), oz = ftd::cload(&g->org[2], 0);
        S.inv_s = ftd::cload(&g->inv_s, 0);
        if (RECORDS) {
            S.org[0] = ox;
            S.org[1] = oy;
            S.org[2] = oz;
        }
        wave_lds_sync();                               // the wave's last tile is done with its LDS
        lds.px[lane] = F.x;
        lds.py[lane] = F.y;
        lds.pz[lane] = F.z;
        lds.best[lane] = none;
        if (MODE == 1) lds.sec[lane] = none;
        // the middle of the tile's first and last node
        auto middle = [](float v) {
            return 0.5f * (__int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0)) +
                           __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63)));
        };
        S.cen[0] = middle(F.x);
        S.cen[1] = middle(F.y);
        S.cen[2] = middle(F.z);
        // one that is not finite, or too large to square: any node that is neither
        // (crossing points are taken about the centre, which must not hide them
        // from the tile's other nodes; its own distances overflow the same way)
        auto usable = [](float u, float v, float w) { return fabsf(u) < 1e18f && fabsf(v) < 1e18f && fabsf(w) < 1e18f; };
        if (!usable(S.cen[0], S.cen[1], S.cen[2])) {
            const uint64_t fin = __ballot(usable(F.x, F.y, F.z));
            const int l = fin ? __ffsll((unsigned long long)fin) - 1 : 0;
            S.cen[0] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(F.x), l));
            S.cen[1] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(F.y), l));
            S.cen[2] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(F.z), l));
        }
        wave_lds_sync();
        const int k = lane >> 4;
#pragma unroll
        for (int cb = 0; cb < 4; cb++) {
            const int j = 16 * cb + (lane & 15);
            if (MODE == 0)
                S.rel[cb] = k == 0 ? lds.px[j] - S.cen[0] : k == 1 ? lds.py[j] - S.cen[1] : k == 2 ? lds.pz[j] - S.cen[2] : 1.0f;
            // rows k = 0, 2 take the coordinates' upper halves (and 1), 1 and 3 the lower
            const Row r = make_row((lds.px[j] - ox) * S.inv_s, (lds.py[j] - oy) * S.inv_s, (lds.pz[j] - oz) * S.inv_s, 1.0f);
            S.B[cb] = (k & 1) ? r.lo : r.hi;
        }
        if (MODE == 0) {
            const float dx = F.x - S.cen[0], dy = F.y - S.cen[1], dz = F.z - S.cen[2];
            S.pp = __fmaf_rn(dz, dz, __fmaf_rn(dy, dy, dx * dx)) * (1.0f - 0x1.0p-18f);
        }
        uint32_t start = ~0u;
        if (a.probe) {
            uint32_t s = ~0u;
            // in a narrow band: none beyond the band and the tile's half diagonal
            const float hx = F.x - S.cen[0], hy = F.y - S.cen[1], hz = F.z - S.cen[2];
            const float half = sqrtf(middle(hx * hx + hy * hy + hz * hz));
            const float lim = (a.band + half) * S.inv_s;
            S.seed(root, (S.cen[0] - ox) * S.inv_s, (S.cen[1] - oy) * S.inv_s, (S.cen[2] - oz) * S.inv_s,
                   a.band > 0.0f ? lim * lim : INFINITY, s, start);
            if (s != ~0u) {                            // every node to it
                uint64_t key;
                if (MODE == 0) {
                    const float4 r = ftd::cload(a.prec, s);
                    const float dx = r.x - F.x, dy = r.y - F.y, dz = r.z - F.z;
                    key = cand_key(sqrtf(dx * dx + dy * dy + dz * dz), __float_as_int(r.w));
                } else {
                    const TriRec r = ftd::cload(a.trec, s);
                    key = cand_key(ftd::tri_dist2(F.x, F.y, F.z, r), ftd::tri_id(r));
                }
                if (key < none) lds.best[lane] = key;
            }
        }
        S.refresh();
        S.walk(root, start, split >= 0 ? kSplitParts : 1, split >= 0 ? __builtin_amdgcn_readfirstlane(split % kSplitParts) : 0);
        wave_lds_sync();
        F.bkey = lds.best[lane];
        if (MODE == 1) F.skey = lds.sec[lane];
    }
    if (split >= 0) {                                  // full domain: nothing is clamped
        a.split_out[(int64_t)split * 64 + lane] = make_ulonglong2(F.bkey, F.skey);
        return;
    }
    const bool clamped = node >= 0 && a.band > 0.0f && F.bj() < 0;
    const uint64_t cm = __ballot(clamped);
    if (lane == 0 && a.band > 0.0f) a.clamped[base >> 6] = (uint32_t)__popcll(cm);
    if (node < 0) return;
    if (STATS) record_stats<MODE>(a, F, node, S.st);
    finish_node<MODE>(a, F, node);
}

// Narrow band: the tiles any primitive can reach, 64 tiles per wave: cls 1 and
// a place in the list, from its front those inside the surface (where the
// longest ones are: they start first), from its end the others, counted in
// `count` (inside << 32 | others).
// A tile counts as its box's ball, and is left out only if the boxes of all
// nodes above the leaves (indices below `last`: those, and the leaves of a field
// that has no such nodes) are farther from the centre than the band and the
// radius, both raised well past the rounding of the boxes and of the distances:
// a tile left out would find nothing.  The walk is the search's, with tiles for
// nodes; a tile leaves it at the first box that it reaches.  Latency is all
// its time, so it does not go down to the leaves, which would leave out few
// more (128^3: 123 us, and 37 down to the nodes above them).
// Searching every tile, 95 % of which end at the root's children, took 1.86 ms
// at 256^3 in a 6 h band; this 0.10 ms, and the search of the rest 1.03 to 1.2,
// with the others' epilogue (k_far_tiles) beside it: 0.16 ms of its own, or 0.97
// from its first block to its last where those wait for the search's persistent
// waves to leave.  At 128^3 0.32, now 0.04 and 0.23.
__global__ __launch_bounds__(64) void k_tile_near(QueryArgs a, uint32_t last, uint32_t* cls, int32_t* list,
                                                  unsigned long long* count)
{
    __shared__ WaveLds<1> lds;
    if (halted(a.sc)) return;
    int lane = ftd::lane_id();
    asm volatile("" : "+v"(lane));
    const int64_t n_tiles = a.n_slots / 64;
    const int64_t tile = (int64_t)blockIdx.x * 64 + lane;
    const int64_t mine = tile < n_tiles ? tile : n_tiles - 1;
    float lo[3], hi[3], odd = 0.0f;
    const float* axes[3] = {a.sx, a.sy, a.sz};
#pragma unroll
    for (int k = 0; k < 3; k++) {
        lo[k] = INFINITY;
        hi[k] = -INFINITY;
        const float4* v = reinterpret_cast<const float4*>(axes[k] + 64 * mine);
#pragma unroll 4
        for (int q = 0; q < 16; q++) {
            const float4 u = v[q];
            lo[k] = fminf(lo[k], fminf(fminf(u.x, u.y), fminf(u.z, u.w)));
            hi[k] = fmaxf(hi[k], fmaxf(fmaxf(u.x, u.y), fmaxf(u.z, u.w)));
            odd += 0.0f * ((u.x + u.y) + (u.z + u.w));         // NaN if a coordinate is not finite
        }
    }
    float c[3], ext2 = 0.0f;
    for (int k = 0; k < 3; k++) {
        c[k] = 0.5f * lo[k] + 0.5f * hi[k];
        const float e = 0.5f * (hi[k] - lo[k]);
        ext2 += e * e;
    }
    const bool ok = odd == 0.0f && ext2 < INFINITY;
    const int field = a.tile_field[mine];
    TileSearch<1, false> S(a, lds, lane);
    uint64_t near = __ballot(!ok);
    // one field of the wave's tiles at a time
    for (uint64_t todo = __ballot(ok && tile < n_tiles); todo;) {
        const int f = __builtin_amdgcn_readlane(field, __ffsll((unsigned long long)todo) - 1);
        const uint64_t here = __ballot(field == f) & todo;
        todo &= ~here;
        const uint32_t root = (uint32_t)__builtin_amdgcn_readfirstlane((int)ftd::cload(a.roots, f));
        if (root == ~0u) continue;                     // the field has no primitives
        const Grid* g = a.grids + f;
        const float ox = ftd::cload(&g->org[0], 0), oy = ftd::cload(&g->org[1], 0), oz = ftd::cload(&g->org[2], 0);
        const float inv_s = ftd::cload(&g->inv_s, 0);
        const bool in = __builtin_amdgcn_inverse_ballot_w64(here);
        const float lim = (a.band + sqrtf(ext2)) * inv_s * (1.0f + 0x1.0p-12f) + 0x1.0p-16f;
        wave_lds_sync();
        lds.px[lane] = in ? (c[0] - ox) * inv_s : 0.0f;
        lds.py[lane] = in ? (c[1] - oy) * inv_s : 0.0f;
        lds.pz[lane] = in ? (c[2] - oz) * inv_s : 0.0f;
        lds.thr[lane] = in ? lim * lim : -1.0f;
        wave_lds_sync();
#pragma unroll
        for (int cb = 0; cb < 4; cb++) {
            const int j = 16 * cb + (lane & 15);
            const Row r = make_row(lds.px[j], lds.py[j], lds.pz[j], 1.0f);
            S.B[cb] = ((lane >> 4) & 1) ? r.lo : r.hi;
            S.thr[cb] = lds.thr[j];
        }
        uint32_t c0 = ftd::cload(a.first, root), c1 = ftd::cload(a.first, root + 1);
        int sp = 0;                                    // list sp: the children of a node
        for (;;) {
            uint32_t f0 = c0;
            uint64_t mask;
            if (f0 < last) {
                near |= S.reached(c0, c1 - c0);
                if (!(here & ~near)) break;
                mask = 0;
            } else {
                mask = S.admitted(c0, c1 - c0, sp);
            }
            while (!mask && sp > 0) {                  // back to a list with something left
                sp--;
                const uint4 t = lds.stack[sp];
                f0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)t.x);
                mask = (uint32_t)__builtin_amdgcn_readfirstlane((int)t.y) |
                       ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)t.z) << 32);
            }
            if (!mask) break;
            const uint32_t b = (uint32_t)(__ffsll((unsigned long long)mask) - 1);
            mask &= mask - 1;
            S.range_of(sp, b, c0, c1);
            if (lane == 0) lds.stack[sp] = make_uint4(f0, (uint32_t)mask, (uint32_t)(mask >> 32), 0u);
            sp++;
        }
    }
    const bool reach = tile < n_tiles && ((near >> lane) & 1ull);
    const bool inside = reach && a.phi_old[a.perm[64 * mine]] < 0.0;   // (a tile's first slot is a node)
    if (tile < n_tiles) cls[tile] = reach;
    const uint64_t m2 = __ballot(inside), m1 = __ballot(reach && !inside), below = (1ull << lane) - 1ull;
    if (!(m1 | m2)) return;
    uint64_t at = 0;
    if (lane == 0) at = atomicAdd(count, ((unsigned long long)__popcll(m2) << 32) | (unsigned long long)__popcll(m1));
    const uint32_t a2 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(at >> 32)), a1 = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
    if (inside) list[a2 + (uint32_t)__popcll(m2 & below)] = (int32_t)tile;
    else if (reach) list[n_tiles - 1 - (int64_t)(a1 + (uint32_t)__popcll(m1 & below))] = (int32_t)tile;
}

// Narrow band: the epilogue of the tiles that no primitive reaches (cls 0), one
// per wave.
template <int MODE>
__global__ __launch_bounds__(kBS) void k_far_tiles(QueryArgs a, const uint32_t* cls)
{
    if (halted(a.sc)) return;
    const int64_t tile = ((int64_t)blockIdx.x * kBS + threadIdx.x) >> 6;
    if (tile >= a.n_slots / 64 || cls[tile]) return;   // whole wave
    const int lane = threadIdx.x & 63;
    const int32_t node = a.perm[tile * 64 + lane];
    const uint64_t m = __ballot(node >= 0);
    if (lane == 0) a.clamped[tile] = (uint32_t)__popcll(m);
    if (node < 0) return;
    Found F;
    F.x = F.y = F.z = 0.0f;                            // (of no use without a candidate)
    F.bkey = F.skey = no_key<MODE>(a);
    finish_node<MODE>(a, F, node);
}

// Query schedule of a launch: a persistent grid (as many waves as the device
// holds, or as there are tiles).  The deep tiles (k_tile_deep) come first, a
// very deep one (a.split_out) as kSplitParts parts, and wave w starts with
// the w-th of them; the waves left over start with the first tiles of their
// XCD (XcdShare).  After its first tile a wave takes the deep tiles that no
// wave started with from one counter, then its XCD's from that XCD's, then
// those of the XCDs that have any left, and leaves when none has: the
// counters only grow, so every wave does.  Against one wave per tile in a fixed
// order, which the dispatcher starts as places get free but on a fixed XCD:
// triangles at 256^3 6.55 -> 6.2 ms, 160 x 144 x 131 1.61 -> 1.55, a 256^3
// band 2.01 -> 1.86; crossing points at 256^3 3.33 -> 3.16; 128^3 and below the
// same.  (Looking at every XCD's counter before each tile cost more than the
// tiles: 8 ms, 5.3 in the band.)
// Launch bound: WPS waves per SIMD.  Six (80 VGPRs, 52 B of spills around
// the FP64 settle) beat five (no spills) and seven at 256^3: triangles 6.79 /
// 6.10 / 6.33 ms at 5 / 6 / 7, points 3.57 / 3.20 / 3.31; the wave's LDS allows
// seven.  The workgroup's size makes little difference, as every wave takes its
// own tiles (a 256^3 step at bins of 1.5: 7.33 ms with 64 threads, 7.18 with 256).
template <int MODE, int BS, int WPS, bool STATS = false, bool RECORDS = false>
__global__ __launch_bounds__(BS, WPS) void k_query_wave(QueryArgs a)
{
    constexpr uint32_t wpb = BS / 64;
    __shared__ WaveLds<MODE> wlds[wpb];
    if (halted(a.sc)) return;                         // an earlier stage failed: phi untouched
    const uint32_t w = threadIdx.x >> 6, xcd = blockIdx.x % kXcds;
    bool more_deep = true;                            // some that no wave started with
    uint32_t from = 0;                                // the XCD after this one by `from` has some left
    for (bool first = true;; first = false) {
        // in a narrow band only the tiles that a primitive can reach, as they come
        const uint64_t listed = a.tile_list ? ftd::cload(a.n_deep, 0) : 0ull;
        const uint32_t inside = (uint32_t)(listed >> 32);
        const uint32_t n_tiles = a.band > 0.0f ? inside + (uint32_t)listed : (uint32_t)(a.n_slots / 64);
        const uint64_t nd = a.band > 0.0f ? 0ull : listed;
        const uint32_t K = (uint32_t)nd, cap = (uint32_t)split_tiles_cap(n_tiles);
        const uint32_t K2 = !a.split_out ? 0u : (uint32_t)(nd >> 32) < cap ? (uint32_t)(nd >> 32) : cap;
        const uint32_t D = K2 * kSplitParts + (K - K2);               // deep parts and tiles
        const uint32_t Db = (D + wpb - 1) / wpb;                      // workgroups that start with them
        const XcdShare share(n_tiles - K);
        // tiles of XCD x that its waves start with
        auto started = [&](uint32_t x) {
            const uint32_t b0 = Db + ((x - Db) & (kXcds - 1));        // its first workgroup after those
            return b0 < gridDim.x ? ((gridDim.x - b0 + kXcds - 1) / kXcds) * wpb : 0u;
        };
        uint32_t deep = ~0u, x = xcd, k = ~0u;                        // the deep-th, or XCD x's k-th
        if (first) {
            if (blockIdx.x < Db) {
                deep = blockIdx.x * wpb + w;
                if (deep >= D) continue;
            } else {
                k = (blockIdx.x - (Db + ((xcd - Db) & (kXcds - 1)))) / kXcds * wpb + w;
                if (k >= share.tiles(xcd)) continue;
            }
        } else {
            more_deep = more_deep && gridDim.x * wpb < D;
            if (more_deep) {
                uint32_t got = 0;
                if (ftd::lane_id() == 0) got = atomicAdd(a.queue, 1u);
                deep = gridDim.x * wpb + (uint32_t)__builtin_amdgcn_readfirstlane((int)got);
                more_deep = deep < D;
            }
            if (!more_deep) {
                deep = ~0u;
                for (; from < kXcds; from++) {
                    x = (xcd + from) % kXcds;
                    const uint32_t nx = share.tiles(x), sx = started(x);
                    if (sx >= nx) continue;
                    uint32_t got = 0;
                    if (ftd::lane_id() == 0) got = atomicAdd(a.queue + kQueueLine * (1 + x), 1u);
                    k = sx + (uint32_t)__builtin_amdgcn_readfirstlane((int)got);
                    if (k < nx) break;
                }
                if (from == kXcds) return;
            }
        }
        int split = -1;
        uint32_t r;                                                   // place in the launch order
        if (deep != ~0u) {
            r = K2 + (deep - K2 * kSplitParts);
            if (deep < K2 * kSplitParts) {
                split = (int)deep;
                r = deep / kSplitParts;
            }
        } else {
            r = K + share.tile(x, k);
            if (a.band > 0.0f && r >= inside) r = (uint32_t)(a.n_slots / 64) - 1u - (r - inside);   // (k_tile_near)
        }
        // the wave's tile as uniform values
        const int64_t tile = __builtin_amdgcn_readfirstlane(a.tile_list ? a.tile_list[r] : (int)r);
        search_tile<MODE, STATS, RECORDS>(a, tile * 64, wlds[w], __builtin_amdgcn_readfirstlane(split));
    }
}

// Clamped nodes per field from the tiles' counts, kClampRun tiles per wave.
// (Counted by one atomic per tile on the field's counter, these atomics, served
// one at a time, took 1.4 of a 256^3 band query's 3.4 ms, 0.2 of 0.5 at 128^3.)
constexpr int kClampRun = 1024;
__global__ __launch_bounds__(kBS) void k_clamp_sum(int64_t n_tiles, const uint32_t* clamped, const int32_t* tile_field,
                                                   unsigned long long* n_clamped, const uint64_t* sc)
{
    if (halted(sc)) return;
    const int64_t t0 = ((int64_t)blockIdx.x * kBS + threadIdx.x) / 64 * kClampRun;
    if (t0 >= n_tiles) return;                         // whole wave
    const int64_t t1 = t0 + kClampRun < n_tiles ? t0 + kClampRun : n_tiles;
    const int lane = threadIdx.x & 63, f0 = tile_field[t0];
    const bool one = tile_field[t1 - 1] == f0;         // (fields own consecutive tiles)
    uint32_t n = 0;
    for (int64_t t = t0 + lane; t < t1; t += 64) {
        if (one) n += clamped[t];
        else if (clamped[t]) atomicAdd(&n_clamped[tile_field[t]], (unsigned long long)clamped[t]);
    }
    for (int o = 32; o >= 1; o >>= 1) n += __shfl_xor(n, o);
    if (one && lane == 0 && n) atomicAdd(&n_clamped[f0], (unsigned long long)n);
}

// The parts of each split tile combined, one wave per tile: per lane the
// least key and the least key other than it over the parts' best and second
// keys, then the node's epilogue.  A part's two differ.  A triangle is tested by
// one part only, the one owning its leaf, but for the seed, which every part
// starts with: the same key from several parts counts once (k1, k2 are keys
// other than the least).  Every triangle that can be the best or a second within
// the FP64 settle's margin is tested by its part: a part prunes with its own
// best, which is no better than the tile's.
template <int MODE>
__global__ __launch_bounds__(kBS) void k_split_merge(QueryArgs a)
{
    if (halted(a.sc)) return;
    const int64_t n_tiles = a.n_slots / 64;
    const int64_t k = ((int64_t)blockIdx.x * kBS + threadIdx.x) >> 6;
    const int64_t cap = split_tiles_cap(n_tiles), nd2 = (int64_t)(ftd::cload(a.n_deep, 0) >> 32);
    const int64_t K2 = nd2 < cap ? nd2 : cap;
    if (k >= K2) return;                               // whole wave
    const int lane = threadIdx.x & 63;
    const int64_t slot = (int64_t)a.tile_list[k] * 64 + lane;
    const int32_t node = a.perm[slot];
    const ulonglong2 v = a.split_out[k * kSplitParts * 64 + lane];
    uint64_t best = v.x, second = v.y;
    for (int p = 1; p < kSplitParts; p++) {
        const ulonglong2 u = a.split_out[(k * kSplitParts + p) * 64 + lane];
        // explicit compares: min() of two 64-bit keys would round them
        const uint64_t nb = u.x < best ? u.x : best;
        const uint64_t k1 = best != nb ? best : second, k2 = u.x != nb ? u.x : u.y;
        second = k2 < k1 ? k2 : k1;
        best = nb;
    }
    if (node < 0) return;
    Found F;
    F.x = a.sx[slot]; F.y = a.sy[slot]; F.z = a.sz[slot];
    F.bkey = best;
    F.skey = second;
    finish_node<MODE>(a, F, node);
}

// ============================================================================
// Level-set normals: Assembler::grad / grad_nodes (Assembler.cpp:11-71), the
// last step of LevelSet::resetPhi_ (LevelSet.cpp:451-453)
// ============================================================================
// Node -> tets lists (Mesh3D::p2t, TetraMesh.cpp:84-86, 115-131): counts,
// scan, scatter, then each list sorted to increasing tet id.
// Node -> tets counts and fills with the references of a workgroup's tets
// gathered first in an LDS table keyed by node (consecutive tets share most
// of their nodes): one memory atomic per distinct node of the workgroup
// instead of one per reference.  A reference that finds no slot within
// kN2tProbe probes goes to memory on its own.  The order inside a node's
// list is arbitrary here; k_n2t_sort makes it the tet order.
constexpr int kN2tHash = 1024;            // LDS slots per workgroup (power of 2)
constexpr int kN2tProbe = 16;
__device__ __forceinline__ int n2t_slot(int32_t* key, int32_t v)
{
    uint32_t h = ((uint32_t)v * 2654435761u) >> (32 - 10);
    for (int p = 0; p < kN2tProbe; p++) {
        const int32_t prev = atomicCAS(&key[h], -1, v);
        if (prev == -1 || prev == v) return (int)h;
        h = (h + 1) & (kN2tHash - 1);
    }
    return -1;
}

// twice: raised when a tet names a node twice.
__global__ __launch_bounds__(kBS) void k_n2t_count(const int4* tets, int64_t T, uint32_t* cnt,
                                                   unsigned long long* twice)
{
    static_assert(kN2tHash == 1 << 10, "the slot hash takes 10 bits");
    __shared__ int32_t key[kN2tHash];
    __shared__ uint32_t num[kN2tHash];
    for (int k = threadIdx.x; k < kN2tHash; k += kBS) {
        key[k] = -1;
        num[k] = 0u;
    }
    __syncthreads();
    const int64_t t = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (t < T) {
        const int4 q = tets[t];
        const int32_t v[4] = {q.x, q.y, q.z, q.w};
        if (q.x == q.y || q.x == q.z || q.x == q.w || q.y == q.z || q.y == q.w || q.z == q.w) *twice = 1ull;
        for (int j = 0; j < 4; j++) {
            const int sl = n2t_slot(key, v[j]);
            if (sl >= 0) atomicAdd(&num[sl], 1u);
            else atomicAdd(&cnt[v[j]], 1u);
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kN2tHash; k += kBS)
        if (key[k] >= 0) atomicAdd(&cnt[key[k]], num[k]);
}

__global__ __launch_bounds__(kBS) void k_n2t_fill(const int4* tets, int64_t T, const uint64_t* off,
                                                  uint32_t* cursor, int32_t* ids)
{
    __shared__ int32_t key[kN2tHash];
    __shared__ uint32_t num[kN2tHash];
    __shared__ uint32_t base[kN2tHash];
    for (int k = threadIdx.x; k < kN2tHash; k += kBS) {
        key[k] = -1;
        num[k] = 0u;
    }
    __syncthreads();
    const int64_t t = (int64_t)blockIdx.x * kBS + threadIdx.x;
    int32_t v[4] = {-1, -1, -1, -1};
    int sl[4] = {-1, -1, -1, -1};
    if (t < T) {
        const int4 q = tets[t];
        v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
        for (int j = 0; j < 4; j++) {
            sl[j] = n2t_slot(key, v[j]);
            if (sl[j] >= 0) atomicAdd(&num[sl[j]], 1u);
        }
    }
    __syncthreads();
    // one reservation per distinct node of the workgroup
    for (int k = threadIdx.x; k < kN2tHash; k += kBS) {
        if (key[k] >= 0) base[k] = atomicAdd(&cursor[key[k]], num[k]);
        num[k] = 0u;                                    // now the slot's local cursor
    }
    __syncthreads();
    if (t < T) {
        for (int j = 0; j < 4; j++) {
            const uint32_t r = sl[j] >= 0 ? base[sl[j]] + atomicAdd(&num[sl[j]], 1u) : atomicAdd(&cursor[v[j]], 1u);
            ids[off[v[j]] + r] = (int32_t)t;
        }
    }
}

// Each node's list sorted to increasing tet id: lists of up to kN2tReg ids in
// registers by a bitonic network (padding sorts last), longer ones in place by
// insertion.
constexpr int kN2tReg = 32;
__global__ __launch_bounds__(kBS) void k_n2t_sort(const uint64_t* off, int64_t N, int32_t* ids)
{
    const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (i >= N) return;
    const uint64_t b = off[i], e = off[i + 1];
    const int n = (int)(e - b);
    if (n <= kN2tReg) {
        int32_t v[kN2tReg];
#pragma unroll
        for (int a = 0; a < kN2tReg; a++) v[a] = a < n ? ids[b + a] : INT32_MAX;
#pragma unroll
        for (int k = 2; k <= kN2tReg; k <<= 1) {
#pragma unroll
            for (int j = k >> 1; j > 0; j >>= 1) {
#pragma unroll
                for (int a = 0; a < kN2tReg; a++) {
                    const int l = a ^ j;
                    if (l > a) {
                        const int32_t x = v[a], y = v[l];
                        const bool sw = (a & k) == 0 ? x > y : x < y;
                        v[a] = sw ? y : x;
                        v[l] = sw ? x : y;
                    }
                }
            }
        }
#pragma unroll
        for (int a = 0; a < kN2tReg; a++)
            if (a < n) ids[b + a] = v[a];
        return;
    }
    for (uint64_t a = b + 1; a < e; a++) {
        const int32_t key = ids[a];
        uint64_t j = a;
        while (j > b && ids[j - 1] > key) { ids[j] = ids[j - 1]; j--; }
        ids[j] = key;
    }
}

// Assembler::grad: per tet, B = [p1-p0, p2-p0, p3-p0] in FP64 from the float
// nodes; its inverse transposed is cofactor(r,c) / det, det = sum of
// cofactor(r,0) B(r,0) as x0 + (x1 + x2) (getElementInfo_ij_,
// Assembler.hpp:429-459); the basis gradients (-1,-1,-1), e1, e2, e3
// (Tetrahedron.hpp:36-50) mapped by it, the first summed left to right; then
// g = ((u0 c0 + u1 c1) + u2 c2) + u3 c3, cast to float.  A singular tet (det
// 0, which the reference only reports) gets a zero gradient.
__global__ __launch_bounds__(kBS) void k_tet_grad(const int4* tets, int64_t T, const float* xyz,
                                                  const double* u, float4* grad_t, const uint64_t* sc)
{
    const int64_t t = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (t >= T || halted(sc)) return;
    const int4 q = tets[t];
    const int qi[4] = {q.x, q.y, q.z, q.w};
    double x[4][3];
    for (int j = 0; j < 4; j++)
        for (int k = 0; k < 3; k++) x[j][k] = (double)xyz[3 * (int64_t)qi[j] + k];
    double B[3][3];
    for (int r = 0; r < 3; r++)
        for (int c = 0; c < 3; c++) B[r][c] = x[c + 1][r] - x[0][r];
    double C[3][3];
    for (int r = 0; r < 3; r++)
        for (int c = 0; c < 3; c++) {
            const int r1 = (r + 1) % 3, r2 = (r + 2) % 3, c1 = (c + 1) % 3, c2 = (c + 2) % 3;
            C[r][c] = B[r1][c1] * B[r2][c2] - B[r1][c2] * B[r2][c1];
        }
    const double det = C[0][0] * B[0][0] + (C[1][0] * B[1][0] + C[2][0] * B[2][0]);
    float g[3] = {0.0f, 0.0f, 0.0f};
    if (det != 0.0) {
        const double inv = 1.0 / det;
        const double u0 = u[qi[0]], u1 = u[qi[1]], u2 = u[qi[2]], u3 = u[qi[3]];
        for (int r = 0; r < 3; r++) {
            const double b0 = C[r][0] * inv, b1 = C[r][1] * inv, b2 = C[r][2] * inv;
            const double c0 = (b0 * -1.0 + b1 * -1.0) + b2 * -1.0;
            g[r] = (float)(((u0 * c0 + u1 * b0) + u2 * b1) + u3 * b2);
        }
    }
    grad_t[t] = make_float4(g[0], g[1], g[2], 0.0f);
}

// The block of nodes of this workgroup: each of the chip's eight dies, which
// get workgroups in turn, has one range of the node numbers to itself, so that
// the gradients that neighbouring nodes share are fetched once into its L2.
__device__ __forceinline__ int64_t die_block()
{
    const uint32_t per = (gridDim.x + 7) / 8;
    const uint32_t full = gridDim.x % 8 == 0 ? 8 : gridDim.x % 8, die = blockIdx.x % 8;
    return (int64_t)die * per - (die > full ? die - full : 0) + blockIdx.x / 8;
}

// Sum of a node's tet gradients in list order.  The loads bound it (nodes of a
// wave share tets only by chance of the numbering), so they are few and in
// flight together: a gradient is one 16-byte load (padded to four floats), the
// list entries come four to a load, and kNodeGather tets are taken at a time.
// Three 4-byte loads a gradient and one an entry took 0.53 ms at
// 160 x 144 x 131; this 0.385 ms, and 0.305 ms with die_block() above, where
// reading the lists and the gradients once at a large copy's rate takes 0.14.
// The list array holds kNodeGather more entries than there are.
constexpr int kNodeGather = 8;
__device__ __forceinline__ void sum_gradients(const int32_t* ids, uint64_t b, uint64_t e, const float4* grad_t, float n[3])
{
    n[0] = n[1] = n[2] = 0.0f;
    for (uint64_t j0 = b; j0 < e; j0 += kNodeGather) {
        int32_t t[kNodeGather];
        memcpy(t, ids + j0, sizeof t);
        float4 g[kNodeGather];
#pragma unroll
        for (int u = 0; u < kNodeGather; u++) {
            g[u] = grad_t[j0 + u < e ? t[u] : t[0]];
        }
#pragma unroll
        for (int u = 0; u < kNodeGather; u++)
            if (j0 + u < e) {
                n[0] += g[u].x;
                n[1] += g[u].y;
                n[2] += g[u].z;
            }
    }
}

// Assembler::grad_nodes: per node, the float mean of its tets' gradients,
// summed in increasing tet id.
__global__ __launch_bounds__(kBS) void k_node_normals(const uint64_t* off, const int32_t* ids,
                                                      const float4* grad_t, int64_t N, float* out,
                                                      const uint64_t* sc)
{
    const int64_t i = die_block() * kBS + threadIdx.x;
    if (i >= N || halted(sc)) return;
    const uint64_t b = off[i], e = off[i + 1];
    float n[3];
    sum_gradients(ids, b, e, grad_t, n);
    const float cnt = (float)(e - b);
    out[3 * i] = n[0] / cnt;
    out[3 * i + 1] = n[1] / cnt;
    out[3 * i + 2] = n[2] / cnt;
}

// ---- interface curvature (LevelSet::getInterfaceCurvature, LevelSet.cpp:215-253)
// g / |g| per node in float (|g| = sqrt(x^2 + (y^2 + z^2)), g_x, g_y, g_z of
// :224-230).  The fields are doubles that hold float values: they are kept as
// floats, four to a node, and widened where they are used.
__global__ __launch_bounds__(kBS) void k_unit_split(const float* g, int64_t N, float4* unit)
{
    const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (i >= N) return;
    const float x = g[3 * i], y = g[3 * i + 1], z = g[3 * i + 2];
    const float nrm = sqrtf(x * x + (y * y + z * z));
    unit[i] = make_float4(x / nrm, y / nrm, z / nrm, 0.0f);
}

// The curvature's gradients (LevelSet.cpp:233-235, the entries :238 uses):
// for c = x, y, z the c-th entry of
// the P1 gradient of g_c, in k_tet_grad's frame and operation order, with one
// frame per tet for the three fields instead of one pass per field.  Gathers
// bound it: one 16-byte load per corner for the three fields (three 8-byte
// loads of separate fields took 0.24 ms at 160 x 144 x 131, now 0.15).
__global__ __launch_bounds__(kBS) void k_tet_grad_diag(const int4* tets, int64_t T, const float* xyz,
                                                       const float4* unit, float4* out, const uint64_t* sc)
{
    const int64_t t = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (t >= T || halted(sc)) return;
    const int4 q = tets[t];
    const int qi[4] = {q.x, q.y, q.z, q.w};
    double x[4][3];
    for (int j = 0; j < 4; j++)
        for (int k = 0; k < 3; k++) x[j][k] = (double)xyz[3 * (int64_t)qi[j] + k];
    double B[3][3];
    for (int r = 0; r < 3; r++)
        for (int c = 0; c < 3; c++) B[r][c] = x[c + 1][r] - x[0][r];
    double C[3][3];
    for (int r = 0; r < 3; r++)
        for (int c = 0; c < 3; c++) {
            const int r1 = (r + 1) % 3, r2 = (r + 2) % 3, c1 = (c + 1) % 3, c2 = (c + 2) % 3;
            C[r][c] = B[r1][c1] * B[r2][c2] - B[r1][c2] * B[r2][c1];
        }
    const double det = C[0][0] * B[0][0] + (C[1][0] * B[1][0] + C[2][0] * B[2][0]);
    float g[3] = {0.0f, 0.0f, 0.0f};
    if (det != 0.0) {
        const double inv = 1.0 / det;
        float uf[4][3];
        for (int j = 0; j < 4; j++) {
            const float4 f = unit[qi[j]];
            uf[j][0] = f.x;
            uf[j][1] = f.y;
            uf[j][2] = f.z;
        }
        for (int r = 0; r < 3; r++) {
            const double u0 = uf[0][r], u1 = uf[1][r], u2 = uf[2][r], u3 = uf[3][r];
            const double b0 = C[r][0] * inv, b1 = C[r][1] * inv, b2 = C[r][2] * inv;
            const double c0 = (b0 * -1.0 + b1 * -1.0) + b2 * -1.0;
            g[r] = (float)(((u0 * c0 + u1 * b0) + u2 * b1) + u3 * b2);
        }
    }
    out[t] = make_float4(g[0], g[1], g[2], 0.0f);
}

// Node curvature (LevelSet.cpp:237-239): per component the float mean over the node's
// tets in increasing id (grad_nodes), then the sum x + y + z in that order.
__global__ __launch_bounds__(kBS) void k_node_div(const uint64_t* off, const int32_t* ids, const float4* gd,
                                                  int64_t N, float* k)
{
    const int64_t i = die_block() * kBS + threadIdx.x;
    if (i >= N) return;
    const uint64_t b = off[i], e = off[i + 1];
    float s[3];
    sum_gradients(ids, b, e, gd, s);
    const float cnt = (float)(e - b);
    const float m0 = s[0] / cnt, m1 = s[1] / cnt, m2 = s[2] / cnt;
    k[i] = (m0 + m1) + m2;
}

// Curvature at the crossing points (:243-250): t = float(phi0 / (phi0 - phi1))
// from the blended phi, then (1.0 - t) k0 in double plus t k1 in float, the
// sum in double rounded to float; in crossing-edge order (e2ifp_).
__global__ __launch_bounds__(kBS) void k_curv_points(const int32_t* ifp2e, int64_t P, const int2* edges,
                                                     const double* phi, const float* k, float* k_if)
{
    const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (i >= P) return;
    const int2 e = edges[ifp2e[i]];
    const float t = (float)(phi[e.x] / (phi[e.x] - phi[e.y]));
    const float tk1 = t * k[e.y];
    k_if[i] = (float)((1.0 - (double)t) * (double)k[e.x] + (double)tk1);
}

// ---- Flow::surfaceTension_ (src/growth/Flow.cpp:307-341) -------------------
// Crossing point i (on edge e = (e0, e1), t = phi[e0] / (phi[e0] - phi[e1])
// as float) adds to node e0 the force (1 - t) st (-k_i) area_i rho n0 and to
// e1 t st (-k_i) area_i rho n1, with n the node's normal over its norm.  The
// reference's loop is an OpenMP loop whose += on a node shared by two points
// races; the result defined here is the serial one, terms added in ascending
// i.  Each node gathers its terms (ids 2i + side, sorted), so the order is
// exact with no atomics on the forces.
__global__ __launch_bounds__(kBS) void k_st_count(const int32_t* ifp2e, int64_t P, const int2* edges,
                                                  uint32_t* cnt)
{
    const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (i >= P) return;
    const int2 e = edges[ifp2e[i]];
    atomicAdd(&cnt[e.x], 1u);
    atomicAdd(&cnt[e.y], 1u);
}

__global__ __launch_bounds__(kBS) void k_st_fill(const int32_t* ifp2e, int64_t P, const int2* edges,
                                                 const uint64_t* off, uint32_t* cursor, int32_t* ids)
{
    const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (i >= P) return;
    const int2 e = edges[ifp2e[i]];
    ids[off[e.x] + atomicAdd(&cursor[e.x], 1u)] = (int32_t)(2 * i);
    ids[off[e.y] + atomicAdd(&cursor[e.y], 1u)] = (int32_t)(2 * i + 1);
}

// Types as the reference evaluates them: (1.0 - t) makes the e0 factor a
// double product, cast to float when it scales the float normal; t * st
// keeps the e1 factor in float; fx is double, each term added as a float.
__global__ __launch_bounds__(kBS) void k_st_apply(const uint64_t* off, const int32_t* ids, int64_t N,
                                                  const int32_t* ifp2e, const int2* edges,
                                                  const double* phi, const float* k, const float* area,
                                                  const float* normals, float st, int32_t rho,
                                                  double* fx, double* fy, double* fz)
{
    const int64_t v = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (v >= N) return;
    const uint64_t b = off[v], e = off[v + 1];
    if (b == e) return;
    const float x = normals[3 * v], y = normals[3 * v + 1], z = normals[3 * v + 2];
    const float nrm = sqrtf(x * x + (y * y + z * z));
    const float nx = x / nrm, ny = y / nrm, nz = z / nrm;
    double ax = fx[v], ay = fy[v], az = fz[v];
    for (uint64_t q = b; q < e; q++) {
        const int32_t id = ids[q];
        const int32_t i = id >> 1;
        const int2 ed = edges[ifp2e[i]];
        const float t = (float)(phi[ed.x] / (phi[ed.x] - phi[ed.y]));
        float sc;
        if ((id & 1) == 0)
            sc = (float)((((1.0 - (double)t) * (double)st) * (double)(-k[i])) * (double)area[i] * (double)rho);
        else
            sc = (((t * st) * (-k[i])) * area[i]) * (float)rho;
        ax += (double)(sc * nx);
        ay += (double)(sc * ny);
        az += (double)(sc * nz);
    }
    fx[v] = ax;
    fy[v] = ay;
    fz[v] = az;
}

// ============================================================================
// Advection (LevelSet::update, LevelSet.cpp:89-141): Crank-Nicolson on the P1
// Galerkin form, (M + s A) phi_n = (M - s A) phi with s = 0.5 dt, solved by
// BiCGSTAB with a Jacobi preconditioner.
//
// Matrices are stored in sliced ELL: slices of kFemSlice rows, each slice
// column-major over its width (the longest row in it), so that a wave reads
// k-th entries of 64 rows in one coalesced access.  Rows keep the reference's
// column order (increasing; Assembler::bilin_with_p2t fills a std::map), and
// every row sum runs over it in that order.
// ============================================================================
constexpr int kFemSlice = 64;          // rows per ELL slice (one wave)
constexpr int kFemMaxCols = 48;        // columns per row (the node and its tet neighbours)

// The four basis functions at the four quadrature points: phi_j is hi at its
// own point, lo0 (j = 0) or lo (j = 1, 2, 3) at the other three.  The points in
// the reference's order are those of j = 1, 2, 3, 0.
struct FemQuad {
    double hi, lo0, lo;
    double w;                          // weight (0.25 / 6)
    __host__ __device__ static constexpr int point(int j) { return (j + 3) & 3; }
    __host__ __device__ double phi(int j, int q) const { return q == point(j) ? hi : j == 0 ? lo0 : lo; }
};

struct FemEll {
    const int32_t* len;                // row lengths
    const uint64_t* soff;              // slice offsets in units of kFemSlice entries
    const int32_t* cols;               // ELL columns (padding: the row itself)
    const int32_t* ndiag;              // per slice: its diagonals, 0 if they are more than kFemDiags
    const int32_t* diag;               // their offsets col - row, ascending, kFemDiags a slice
    const uint32_t* dmask;             // per row: which of its slice's diagonals it has
    int twice;                         // a tet of the mesh names a node twice
};
__device__ __forceinline__ int64_t ell_at(const FemEll& e, int64_t i, int k)
{
    return ((int64_t)e.soff[i / kFemSlice] + k) * kFemSlice + (i % kFemSlice);
}

// Row i's product with y: sum over its entries in column order.  (The solver
// calls it with whole waves on whole slices, so the slice is uniform.)
//
// Memory bounds it.  On a mesh numbered along lines the rows of a slice share
// a few diagonals (col - row), so their columns are one list per slice and a
// mask per row, 6 bytes a row instead of 4 per entry: 8.2 bytes an entry
// instead of 12.3.  A slice with more than kFemDiags (a numbering without
// such lines) reads its columns.  At 200^3 0.27-0.28 ms a
// product (4.3 TB/s, a large copy's rate) after 0.37 with 12.3 bytes an entry;
// groups of 4 or 16 diagonals are within 1 % of 8, and parts of the rows kept
// to one die's L2 (as die_block()) took 0.30.
constexpr int kFemDiags = 32;                          // bits of a row's mask
constexpr int kFemGroup = 8;                           // diagonals whose loads are in flight together
__device__ __forceinline__ double ell_dot(const FemEll& e, const double* __restrict__ vals,
                                          const double* __restrict__ y, int64_t i)
{
    const int64_t slice = __builtin_amdgcn_readfirstlane((int)(i / kFemSlice));
    const double* __restrict__ l = vals + (int64_t)e.soff[slice] * kFemSlice + (i % kFemSlice);
    const int nd = e.ndiag[slice];
    double t = 0.0;
    if (nd > 0) {
        const int32_t* __restrict__ dg = e.diag + slice * kFemDiags;
        const uint32_t m = e.dmask[i];
        for (int d0 = 0; d0 < nd; d0 += kFemGroup) {
            double a[kFemGroup], b[kFemGroup];
#pragma unroll
            for (int u = 0; u < kFemGroup; u++) {
                a[u] = b[u] = 0.0;
                if ((m >> (d0 + u)) & 1u) {            // no bit is set past nd
                    a[u] = *l;
                    b[u] = y[i + dg[d0 + u]];
                    l += kFemSlice;
                }
            }
#pragma unroll
            for (int u = 0; u < kFemGroup; u++)
                if ((m >> (d0 + u)) & 1u) t += a[u] * b[u];
        }
    } else {
        const int32_t* __restrict__ c = e.cols + (l - vals);
        const int len = e.len[i];
        for (int k = 0; k < len; k++) t += l[(int64_t)k * kFemSlice] * y[c[(int64_t)k * kFemSlice]];
    }
    return t;
}

// getElementInfo_ij_ (Assembler.hpp:429-459) and the mapped basis gradients
// G[j] = invBt grad(phi_j) (the constant gradients (-1,-1,-1), e1, e2, e3,
// Tetrahedron.hpp:36-50; sums left to right, as in k_tet_grad).  False for a
// singular map, whose tet the reference leaves with an unset inverse.
// x: the tet's four nodes, in its local order.
__device__ __forceinline__ bool fem_frame(const double x[4][3], double G[4][3], double& detB)
{
    double B[3][3], C[3][3];
    for (int r = 0; r < 3; r++)
        for (int c = 0; c < 3; c++) B[r][c] = x[c + 1][r] - x[0][r];
    for (int r = 0; r < 3; r++)
        for (int c = 0; c < 3; c++) {
            const int r1 = (r + 1) % 3, r2 = (r + 2) % 3, c1 = (c + 1) % 3, c2 = (c + 2) % 3;
            C[r][c] = B[r1][c1] * B[r2][c2] - B[r1][c2] * B[r2][c1];
        }
    const double det = C[0][0] * B[0][0] + (C[1][0] * B[1][0] + C[2][0] * B[2][0]);
    if (det == 0.0) return false;
    const double inv = 1.0 / det;
    for (int r = 0; r < 3; r++) {
        const double b0 = C[r][0] * inv, b1 = C[r][1] * inv, b2 = C[r][2] * inv;
        G[0][r] = (b0 * -1.0 + b1 * -1.0) + b2 * -1.0;
        G[1][r] = b0;
        G[2][r] = b1;
        G[3][r] = b2;
    }
    detB = fabs(det);
    return true;
}

// First position in the sorted lst[0, cnt) whose entry is not below v
// (binary search: most of a row's candidates are already in its list).
__device__ __forceinline__ int fem_lower_bound(const int32_t* lst, int cnt, int32_t v)
{
    int lo = 0, hi = cnt;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (lst[mid] < v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// The tets a0 + u (u < kFemGather, those below a1) of a row's list, their
// list entries and then the tets loaded together: kFemGather of each load in
// flight per lane instead of one dependent pair at a time (at 256^3
// k_fem_rowfill 19.7 ms with one, 9.6 with four, 8.8 with eight).
constexpr int kFemGather = 8;
__device__ __forceinline__ void fem_gather_tets(const int32_t* n2t_ids, const int4* tets, uint64_t a0,
                                                uint64_t a1, int4 (&q)[kFemGather])
{
    int32_t id[kFemGather];
#pragma unroll
    for (int u = 0; u < kFemGather; u++) id[u] = a0 + u < a1 ? n2t_ids[a0 + u] : -1;
#pragma unroll
    for (int u = 0; u < kFemGather; u++) q[u] = id[u] >= 0 ? tets[id[u]] : make_int4(0, 0, 0, 0);
}

// Sorted unique columns of row i (the node and every node of its tets) into
// lst; returns the count, or -1 past kFemMaxCols.
__device__ int fem_row_cols(const uint64_t* n2t_off, const int32_t* n2t_ids, const int4* tets, int64_t i,
                            int32_t* lst)
{
    int cnt = 0;
    const uint64_t a1 = n2t_off[i + 1];
    for (uint64_t a0 = n2t_off[i]; a0 < a1; a0 += kFemGather) {
        int4 q[kFemGather];
        fem_gather_tets(n2t_ids, tets, a0, a1, q);
        for (int u = 0; u < kFemGather && a0 + u < a1; u++) {
            const int v4[4] = {q[u].x, q[u].y, q[u].z, q[u].w};
            for (int j = 0; j < 4; j++) {
                const int32_t v = v4[j];
                const int pos = fem_lower_bound(lst, cnt, v);
                if (pos < cnt && lst[pos] == v) continue;
                if (cnt == kFemMaxCols) return -1;
                for (int k = cnt; k > pos; k--) lst[k] = lst[k - 1];
                lst[pos] = v;
                cnt++;
            }
        }
    }
    return cnt;
}

// Pass 1 of the pattern: row lengths and slice widths.  One wave per slice.
__global__ __launch_bounds__(kFemSlice) void k_fem_rowlen(const uint64_t* n2t_off, const int32_t* n2t_ids,
                                                          const int4* tets, int64_t N, int32_t* len,
                                                          uint32_t* width, unsigned* flags)
{
    __shared__ int32_t lst[kFemSlice][kFemMaxCols + 1];
    const int64_t i = (int64_t)blockIdx.x * kFemSlice + threadIdx.x;
    int cnt = 0;
    if (i < N) {
        cnt = fem_row_cols(n2t_off, n2t_ids, tets, i, lst[threadIdx.x]);
        if (cnt < 0) { atomicOr(&flags[0], 1u); cnt = 0; }
        len[i] = cnt;
    }
    int wmax = cnt;
    for (int o = 32; o >= 1; o >>= 1) wmax = max(wmax, __shfl_xor(wmax, o));
    if (threadIdx.x == 0) {
        width[blockIdx.x] = (uint32_t)wmax;
        atomicMax(&flags[1], (unsigned)wmax);                // longest row of the mesh
    }
}

// Pass 2: the ELL columns (padding entries name the row itself) and the
// scatter map: for the a-th tet of row i (n2t order), the row positions of
// its four nodes, one byte each, in fmap[n2t_off[i] + a].
__global__ __launch_bounds__(kFemSlice) void k_fem_rowfill(const uint64_t* n2t_off, const int32_t* n2t_ids,
                                                           const int4* tets, int64_t N, FemEll e,
                                                           const uint32_t* width, int32_t* cols,
                                                           uint32_t* fmap)
{
    __shared__ int32_t lst[kFemSlice][kFemMaxCols + 1];
    const int64_t i = (int64_t)blockIdx.x * kFemSlice + threadIdx.x;
    if (i >= N) return;
    int32_t* l = lst[threadIdx.x];
    const int cnt = fem_row_cols(n2t_off, n2t_ids, tets, i, l);
    const int W = (int)width[blockIdx.x];
    for (int k = 0; k < W; k++) cols[ell_at(e, i, k)] = (k < cnt) ? l[k] : (int32_t)i;
    const uint64_t a1 = n2t_off[i + 1];
    for (uint64_t a0 = n2t_off[i]; a0 < a1; a0 += kFemGather) {
        int4 q[kFemGather];
        fem_gather_tets(n2t_ids, tets, a0, a1, q);
        for (int u = 0; u < kFemGather && a0 + u < a1; u++) {
            const int v4[4] = {q[u].x, q[u].y, q[u].z, q[u].w};
            uint32_t m = 0;
            for (int j = 0; j < 4; j++) {
                // every node of the row's tets is in its list (cnt >= 1 here)
                const int k = fem_lower_bound(l, cnt, v4[j]);
                m |= (uint32_t)(k < cnt ? k : cnt - 1) << (8 * j);
            }
            fmap[a0 + u] = m;
        }
    }
}

// The diagonals of a slice: the rows' ascending offsets merged, the least one
// not yet taken at a time.  One wave per slice.
__global__ __launch_bounds__(kFemSlice) void k_fem_diags(int64_t N, FemEll e, int32_t* ndiag, int32_t* diag,
                                                         uint32_t* dmask)
{
    const int64_t i = (int64_t)blockIdx.x * kFemSlice + threadIdx.x, none = INT64_MAX;
    const int len = i < N ? e.len[i] : 0;
    uint32_t m = 0;
    int k = 0, nd = 0;
    for (;; nd++) {
        const int64_t d = k < len ? (int64_t)e.cols[ell_at(e, i, k)] - i : none;
        int64_t lo = d;
        for (int o = 32; o >= 1; o >>= 1) lo = min(lo, (int64_t)__shfl_xor((long long)lo, o));
        if (lo == none) break;
        if (nd == kFemDiags) { nd = 0; break; }
        if (d == lo) { m |= 1u << nd; k++; }
        if (threadIdx.x == 0) diag[(int64_t)blockIdx.x * kFemDiags + nd] = (int32_t)lo;
    }
    if (i < N) dmask[i] = m;
    if (threadIdx.x == 0) {
        ndiag[blockIdx.x] = nd;
        for (int z = nd; z < kFemDiags; z++) diag[(int64_t)blockIdx.x * kFemDiags + z] = 0;
    }
}

// Rows of the mass (FORM 0) or advection (FORM 1) form of
// Assembler::bilin_with_p2t (Assembler.hpp:131-226): over the tets of row i
// in increasing id and their local nodes j, the integral
// ((f0 w + f2 w) + (f1 w + f3 w)) |det B| of f(u = phi_j, v = phi_i) is
// added to column t(j):  mass  f = u v;  advection  f = V1 (ux v) + V2 (uy v)
// + V3 (uz v) with V_c(q) = sum_j V_c[t(j)] phi_j(q) accumulated from 0 in
// j order (vel: the velocity interleaved per node).
//
// kFemLanes lanes share a row and take its tets in rounds.  First the row's
// columns are gathered once into LDS: each column node's coordinates (and,
// for the advection form, its velocity), so that a tet's nodes are read
// there through its column map (fmap: the row slot of each of its four
// nodes) instead of through the tet list.  Then in each round lane L
// computes the four contributions of tet kFemLanes r + L, and then
// the row's lanes add that round's tets into the row accumulator in tet order,
// lane L the node L of each, so every entry is summed exactly as the
// reference's std::map does.
// A workgroup is one wave of kFemRowsPerWave rows.
constexpr int kFemLanes = 4;
constexpr int kFemRowsPerWave = 64 / kFemLanes;
constexpr int kFemCols = 4;                          // columns per lane whose loads are in flight together
static_assert(kFemLanes == 4, "a row's lanes are a quad (quad_lane, quad_transpose)");

// x of the quad's lane t, in all four.
template <int T>
__device__ __forceinline__ uint32_t quad_lane(uint32_t x)
{
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x55 * T, 0xf, 0xf, true);
}

template <int CTRL>
__device__ __forceinline__ double quad_swap(double x)
{
    const int2 v = __builtin_bit_cast(int2, x);
    return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_mov_dpp(v.x, CTRL, 0xf, 0xf, true),
                                                __builtin_amdgcn_mov_dpp(v.y, CTRL, 0xf, 0xf, true)));
}

// Of a pair that the lanes with and without `up` hold: the one keeps a and
// gets the other's, the other keeps b.
template <int CTRL>
__device__ __forceinline__ void quad_exchange(double& a, double& b, bool up)
{
    const double got = quad_swap<CTRL>(up ? a : b);
    a = up ? got : a;
    b = up ? b : got;
}

// s[j] of lane t becomes s[t] of lane j (t, j: lanes of a quad).
__device__ __forceinline__ void quad_transpose(double (&s)[4], int lane)
{
    quad_exchange<0xB1>(s[0], s[1], lane & 1);        // quad_perm [1, 0, 3, 2]
    quad_exchange<0xB1>(s[2], s[3], lane & 1);
    quad_exchange<0x4E>(s[0], s[2], lane & 2);        // quad_perm [2, 3, 0, 1]
    quad_exchange<0x4E>(s[1], s[3], lane & 2);
}

// LDS per wave, in this order: kFemRowsPerWave accumulators of `stride`
// doubles; for the advection form the column velocities (3 doubles per column
// slot); the column coordinates (3 floats per slot); the row's own slot (one
// word per row).  The velocity region is free after the rounds: k_fem_cn
// reuses it.
__host__ __device__ inline size_t fem_lds_bytes(int stride, int form)
{
    const size_t R = kFemRowsPerWave, S = (size_t)stride;
    return 8 * R * S + (form == 1 ? 24 * R * S : 0) + 12 * R * S + 4 * R;
}

template <int FORM>
struct FemLds {
    double* acc;       // the row's accumulator
    double* vel;       // the row's column velocities (FORM 1)
    float* xyz;        // the row's column coordinates
    int* own;          // the row's own slot
    __device__ FemLds(double* lds, int stride, int rl)
    {
        const size_t R = kFemRowsPerWave, S = (size_t)stride;
        acc = lds + rl * S;
        double* v0 = lds + R * S;
        vel = v0 + rl * 3 * S;
        float* x0 = reinterpret_cast<float*>(v0 + (FORM == 1 ? 3 * R * S : 0));
        xyz = x0 + rl * 3 * S;
        own = reinterpret_cast<int*>(x0 + 3 * R * S) + rl;
    }
};

template <int FORM>
__device__ void fem_rows(const uint64_t* __restrict__ n2t_off, const uint32_t* __restrict__ fmap,
                         const float* __restrict__ xyz, const double* __restrict__ vel, int64_t N,
                         const FemQuad& qd, const FemEll& e, int stride, double* lds, int64_t& row, double*& acc,
                         int& len)
{
    const int lane = threadIdx.x % kFemLanes, rl = threadIdx.x / kFemLanes;
    const int64_t i = (int64_t)blockIdx.x * kFemRowsPerWave + rl;
    const FemLds<FORM> L(lds, stride, rl);
    acc = L.acc;
    row = i;
    len = 0;
    uint64_t a0 = 0;
    int na = 0;
    if (i < N) {
        a0 = n2t_off[i];
        na = (int)(n2t_off[i + 1] - a0);
        len = e.len[i];
        for (int k0 = lane; k0 < len; k0 += kFemCols * kFemLanes) {
            int32_t c[kFemCols];
            float cx[kFemCols][3];
            double cv[kFemCols][3];
            for (int u = 0; u < kFemCols; u++) c[u] = e.cols[ell_at(e, i, min(k0 + kFemLanes * u, len - 1))];
            for (int u = 0; u < kFemCols; u++)
                for (int d = 0; d < 3; d++) {
                    cx[u][d] = xyz[3 * (int64_t)c[u] + d];
                    cv[u][d] = FORM == 1 ? vel[3 * (int64_t)c[u] + d] : 0.0;
                }
            for (int u = 0; u < kFemCols; u++) {
                const int k = k0 + kFemLanes * u;
                if (k >= len) break;
                for (int d = 0; d < 3; d++) L.xyz[3 * k + d] = cx[u][d];
                if (FORM == 1)
                    for (int d = 0; d < 3; d++) L.vel[3 * k + d] = cv[u][d];
                if (c[u] == (int32_t)i) *L.own = k;
                acc[k] = 0.0;
            }
        }
    }
    int na_max = na;                                   // rounds are uniform over the wave
    for (int o = 32; o >= 1; o >>= 1) na_max = max(na_max, __shfl_xor(na_max, o));
    uint32_t mn = lane < na ? fmap[a0 + lane] : 0u;    // maps one round ahead
    __syncthreads();
    const int own = i < N ? *L.own : 0;
    for (int r0 = 0; r0 < na_max; r0 += kFemLanes) {
        const int a = r0 + lane;
        const uint32_t mp = mn;
        if (a + kFemLanes < na) mn = fmap[a0 + a + kFemLanes];
        double add[4] = {0.0, 0.0, 0.0, 0.0};
        if (a < na) {
            int sl[4];
            double x[4][3];
            for (int j = 0; j < 4; j++) {
                sl[j] = (int)((mp >> (8 * j)) & 0xffu);
                for (int d = 0; d < 3; d++) x[j][d] = (double)L.xyz[3 * sl[j] + d];
            }
            double G[4][3], detB;
            if (fem_frame(x, G, detB)) {               // else no contribution
                const int li = sl[0] == own ? 0 : sl[1] == own ? 1 : sl[2] == own ? 2 : 3;
                // quadrature points in the order 0, 2, 1, 3: s02 = f0 w + f2 w and
                // s13 = f1 w + f3 w per basis function, then (s02 + s13) |det B|
                const double w = qd.w;
                double V[4][3];                        // the velocity at the points, summed in node order
                if (FORM == 1)
                    for (int d = 0; d < 3; d++) {
                        // a node's velocity has two products over the four points (hi, lo); a
                        // sum starts with its first product (the reference's 0.0 + that only
                        // turns -0 into +0, which no sum of the row can tell: it starts at +0)
                        double lo[4], hi[4];
                        for (int j = 0; j < 4; j++) {
                            const double vj = L.vel[3 * sl[j] + d];
                            lo[j] = vj * (j == 0 ? qd.lo0 : qd.lo);
                            hi[j] = vj * qd.hi;
                        }
                        const double l01 = lo[0] + lo[1];
                        V[0][d] = ((lo[0] + hi[1]) + lo[2]) + lo[3];
                        V[1][d] = (l01 + hi[2]) + lo[3];
                        V[2][d] = (l01 + lo[2]) + hi[3];
                        V[3][d] = ((hi[0] + lo[1]) + lo[2]) + lo[3];
                    }
                double s02[4], s13[4];
                for (int qq = 0; qq < 4; qq++) {
                    const int q4 = qq == 1 ? 2 : qq == 2 ? 1 : qq;
                    const double v = q4 == FemQuad::point(li) ? qd.hi : li == 0 ? qd.lo0 : qd.lo;
                    for (int j = 0; j < 4; j++) {
                        const double f = FORM == 0
                            ? qd.phi(j, q4) * v
                            : (V[q4][0] * (G[j][0] * v) + V[q4][1] * (G[j][1] * v)) + V[q4][2] * (G[j][2] * v);
                        const double pw = f * w;
                        if (qq == 0) s02[j] = pw;
                        else if (qq == 1) s02[j] = s02[j] + pw;
                        else if (qq == 2) s13[j] = pw;
                        else s13[j] = s13[j] + pw;
                    }
                }
                for (int j = 0; j < 4; j++) add[j] = (s02[j] + s13[j]) * detB;
            }
        }
        // a tet's four nodes are four distinct columns, unless a tet of the mesh
        // names one twice: each of the row's lanes adds one of them (in turn, then);
        // tets stay in order (the lanes are of one wave, whose LDS operations are
        // done in order)
        quad_transpose(add, lane);
        const uint32_t pos[4] = {quad_lane<0>(mp), quad_lane<1>(mp), quad_lane<2>(mp), quad_lane<3>(mp)};
        if (!e.twice) {
            for (int t = 0; t < 4; t++) {
                if (r0 + t < na) acc[(pos[t] >> (8 * lane)) & 0xffu] += add[t];
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
        } else {
            for (int t = 0; t < 4; t++)
                for (int l = 0; l < kFemLanes; l++) {
                    if (r0 + t < na && lane == l) acc[(pos[t] >> (8 * lane)) & 0xffu] += add[t];
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                }
        }
    }
}

// The velocity interleaved per node (vx, vy, vz), so that a tet's gathers
// touch one 24-byte run per node instead of three arrays.
__global__ __launch_bounds__(kBS) void k_vel_interleave(const double* flow, int64_t N, double* vel3)
{
    const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (i >= N) return;
    vel3[3 * i] = flow[i];
    vel3[3 * i + 1] = flow[N + i];
    vel3[3 * i + 2] = flow[2 * N + i];
}

// The mass matrix, once per mesh (LevelSet::init, LevelSet.cpp:35-39).
__global__ __launch_bounds__(64) void k_fem_mass(const uint64_t* n2t_off, const uint32_t* fmap,
                                                 const float* xyz, int64_t N, FemQuad qd, FemEll e, int stride, double* mvals)
{
    extern __shared__ double fem_lds[];
    int64_t i;
    double* acc;
    int len;
    fem_rows<0>(n2t_off, fmap, xyz, nullptr, N, qd, e, stride, fem_lds, i, acc, len);
    for (int k = threadIdx.x % kFemLanes; k < len; k += kFemLanes) mvals[ell_at(e, i, k)] = acc[k];
}

// The advection matrix alone (ft_fem_assemble), into vals in ELL layout.
__global__ __launch_bounds__(64) void k_fem_adv(const uint64_t* n2t_off, const uint32_t* fmap,
                                                const float* xyz, const double* vel, int64_t N, FemQuad qd, FemEll e, int stride,
                                                double* vals)
{
    extern __shared__ double fem_lds[];
    int64_t i;
    double* acc;
    int len;
    fem_rows<1>(n2t_off, fmap, xyz, vel, N, qd, e, stride, fem_lds, i, acc, len);
    for (int k = threadIdx.x % kFemLanes; k < len; k += kFemLanes) vals[ell_at(e, i, k)] = acc[k];
}

// ELL rows to CSR at the row offsets off (a scan of the lengths).
__global__ __launch_bounds__(kBS) void k_ell_to_csr(int64_t N, FemEll e, const double* vals, const uint64_t* off,
                                                    int32_t* cols, double* out)
{
    const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (i >= N) return;
    const int len = e.len[i];
    for (int k = 0; k < len; k++) {
        const int64_t at = ell_at(e, i, k);
        cols[off[i] + k] = e.cols[at];
        out[off[i] + k] = vals[at];
    }
}

// Deterministic block sum of up to two values per thread into part[2 b], part[2 b + 1].
template <int BS>
__device__ __forceinline__ void block_sum2(double a, double b, double* part)
{
    __shared__ double red[2][BS / 64];
    for (int o = 32; o >= 1; o >>= 1) {
        a += __shfl_xor(a, o);
        b += __shfl_xor(b, o);
    }
    if ((threadIdx.x & 63) == 0) { red[0][threadIdx.x >> 6] = a; red[1][threadIdx.x >> 6] = b; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double sa = 0.0, sb = 0.0;
        for (int w = 0; w < BS / 64; w++) { sa += red[0][w]; sb += red[1][w]; }
        part[2 * blockIdx.x] = sa;
        part[2 * blockIdx.x + 1] = sb;
    }
}

// Per call: the advection row, then L = M + s A and R = M - s A entrywise
// (LevelSet.cpp:126-127), invdiag = 1 / L_ii (1 where 0: Eigen's
// DiagonalPreconditioner), b = R phi and r = b - L phi (BiCGSTAB's first
// residual from the guess phi), each summed in column order; r0 = r, x = phi,
// p = v = 0.
//
// FP64 arithmetic bounds it (about 260 operations per row and tet, none of them
// a matrix product: each row's basis gradients differ), with the latency of LDS
// and of the columns' gathers behind it; LDS holds it at 3 waves per SIMD.  At
// 200^3 3.13 ms, after 4.23: 3.84 with the quadrature's shared products and
// the additions spread over a row's lanes, 3.44 with kFemCols columns' loads in
// flight (one: 3.84), 3.13 with the contributions exchanged between lanes in
// registers instead of LDS.  91 VGPRs; asking for 4 waves changes nothing.
__global__ __launch_bounds__(64, 3) void k_fem_cn(const uint64_t* __restrict__ n2t_off,
                                               const uint32_t* __restrict__ fmap, const float* __restrict__ xyz,
                                               const double* __restrict__ vel, int64_t N, FemQuad qd, FemEll e,
                                               int stride, const double* __restrict__ mvals, double s,
                                               const double* __restrict__ phi, double* __restrict__ lvals,
                                               double* __restrict__ invdiag, double* __restrict__ b,
                                               double* __restrict__ x, double* __restrict__ r,
                                               double* __restrict__ r0, double* __restrict__ p,
                                               double* __restrict__ v)
{
    extern __shared__ double fem_lds[];
    int64_t i;
    double* A;
    int len;
    fem_rows<1>(n2t_off, fmap, xyz, vel, N, qd, e, stride, fem_lds, i, A, len);
    // the row's entries split over its lanes: L = M + s A into lvals, the
    // products R phi_c (in place of A) and L phi_c into LDS; then two lanes
    // sum them in column order, as a sequential row loop would
    const int lane = threadIdx.x % kFemLanes;
    double* LP = FemLds<1>(fem_lds, stride, threadIdx.x / kFemLanes).vel;   // free after the rounds
    double id = 0.0;                                   // L_ii, in the lane that has it
    for (int k0 = lane; k0 < len; k0 += kFemCols * kFemLanes) {
        const int64_t at0 = ell_at(e, i, k0);
        int32_t c[kFemCols];
        double m[kFemCols], pc[kFemCols];
        for (int u = 0; u < kFemCols; u++) {
            const int64_t at = ell_at(e, i, min(k0 + kFemLanes * u, len - 1));
            c[u] = e.cols[at];
            m[u] = mvals[at];
        }
        for (int u = 0; u < kFemCols; u++) pc[u] = phi[c[u]];
        for (int u = 0; u < kFemCols; u++) {
            const int k = k0 + kFemLanes * u;
            if (k >= len) break;
            const double sa = s * A[k];
            const double L = m[u] + sa, R = m[u] - sa;
            lvals[at0 + kFemLanes * kFemSlice * u] = L;
            A[k] = R * pc[u];
            LP[k] = L * pc[u];
            if (c[u] == (int32_t)i) id = L;
        }
    }
    for (int o = 1; o < kFemLanes; o <<= 1) {          // the diagonal to all
        const double vo = __shfl_xor(id, o);
        if (id == 0.0) id = vo;
    }
    __syncthreads();
    // lane 0 sums b_i, lane 1 (L phi)_i, kFemLanes terms read at a time
    const double* S = lane == 0 ? A : LP;
    double sum = 0.0;
    if (lane < 2)
        for (int k0 = 0; k0 < len; k0 += kFemLanes) {
            double a[kFemLanes];
            for (int u = 0; u < kFemLanes; u++) a[u] = S[min(k0 + u, len - 1)];
            for (int u = 0; u < kFemLanes; u++)
                if (k0 + u < len) sum += a[u];
        }
    const double lx = __shfl_xor(sum, 1);
    if (i < N && lane == 0) {
        const double bi = sum, ri = bi - lx;
        invdiag[i] = id != 0.0 ? 1.0 / id : 1.0;
        b[i] = bi;
        x[i] = phi[i];
        r[i] = ri;
        r0[i] = ri;
        p[i] = 0.0;
        v[i] = 0.0;
    }
}

// ---- BiCGSTAB (Eigen's bicgstab; H. A. van der Vorst 1992) ----------------
// Scalars live on the device; each finishing kernel reduces the block
// partials (in block order) and updates them.  stop: the iteration that just
// ended is the last, or needs a restart before the next; the kernels of an
// iteration that was enqueued beyond it do nothing.
struct BcgScalars {
    double rho, rho_old, alpha, w;
    double rr, bb, r0sq;
    double r0v, tt, ts;
    uint64_t stop;
};

constexpr int kBcgBS = 256;
constexpr int kBcgGrid = 2048;         // workgroups of the solver kernels (block partials)
constexpr int kBcgAhead = 2;           // iterations in flight

// Grid-stride loops: row i is handled by workgroup (i / kBcgBS) % gridDim.x;
// each thread sums its rows in order, so the partials are fixed by N and the
// grid size alone.
#define BCG_ROWS(i) for (int64_t i = (int64_t)blockIdx.x * kBcgBS + threadIdx.x; i < N; \
                         i += (int64_t)gridDim.x * kBcgBS)

// The preconditioned vectors y = P p and z = P s (P = invdiag) are formed
// once per row and stored, so that each SpMV entry gathers one value instead
// of forming them from two or three gathers; each is the same product as
// when formed where read.

// p = r + beta (p - w v), beta = (rho / rho_old) (alpha / w); y = invdiag p.
__global__ __launch_bounds__(kBcgBS) void k_bcg_p(int64_t N, const BcgScalars* sc, const double* r,
                                                  const double* v, const double* invdiag, double* p, double* y)
{
    if (sc->stop) return;
    const double beta = (sc->rho / sc->rho_old) * (sc->alpha / sc->w), w = sc->w;
    BCG_ROWS(i) {
        const double pi = r[i] + beta * (p[i] - w * v[i]);
        p[i] = pi;
        y[i] = invdiag[i] * pi;
    }
}

// v = L y (y = P p, then v = A y); partial r0.v.
__global__ __launch_bounds__(kBcgBS) void k_bcg_v(int64_t N, const BcgScalars* sc, FemEll e, const double* lvals,
                                                  const double* y, const double* r0, double* v, double* part)
{
    if (sc->stop) return;
    double d = 0.0;
    BCG_ROWS(i) {
        const double t = ell_dot(e, lvals, y, i);
        v[i] = t;
        d += r0[i] * t;
    }
    block_sum2<kBcgBS>(d, 0.0, part);
}

// s = r - alpha v; z = invdiag s.
__global__ __launch_bounds__(kBcgBS) void k_bcg_s(int64_t N, const BcgScalars* sc, const double* invdiag,
                                                  const double* r, const double* v, double* s_, double* z)
{
    if (sc->stop) return;
    const double alpha = sc->alpha;
    BCG_ROWS(i) {
        const double si = r[i] - alpha * v[i];
        s_[i] = si;
        z[i] = invdiag[i] * si;
    }
}

// t = L z; partials t.t and t.s.
__global__ __launch_bounds__(kBcgBS) void k_bcg_t(int64_t N, const BcgScalars* sc, FemEll e, const double* lvals,
                                                  const double* z, const double* s_, double* t, double* part)
{
    if (sc->stop) return;
    double tt = 0.0, ts = 0.0;
    BCG_ROWS(i) {
        const double acc = ell_dot(e, lvals, z, i);
        t[i] = acc;
        tt += acc * acc;
        ts += acc * s_[i];
    }
    block_sum2<kBcgBS>(tt, ts, part);
}

// x += alpha y + w z;  r = s - w t;  partials r.r and r0.r.
__global__ __launch_bounds__(kBcgBS) void k_bcg_x(int64_t N, const double* y, const double* s_,
                                                  const double* z, const double* t, const double* r0,
                                                  const BcgScalars* sc, double* x, double* r, double* part)
{
    if (sc->stop) return;
    const double alpha = sc->alpha, w = sc->w;
    double rr = 0.0, r0r = 0.0;
    BCG_ROWS(i) {
        x[i] = x[i] + (alpha * y[i] + w * z[i]);
        const double ri = s_[i] - w * t[i];
        r[i] = ri;
        rr += ri * ri;
        r0r += r0[i] * ri;
    }
    block_sum2<kBcgBS>(rr, r0r, part);
}

// Restart (a residual too orthogonal to r0): r = b - L x, r0 = r; partial r.r.
__global__ __launch_bounds__(kBcgBS) void k_bcg_restart(int64_t N, FemEll e, const double* lvals,
                                                        const double* b, const double* x, double* r,
                                                        double* r0, double* part)
{
    double rr = 0.0;
    BCG_ROWS(i) {
        const double ri = b[i] - ell_dot(e, lvals, x, i);
        r[i] = ri;
        r0[i] = ri;
        rr += ri * ri;
    }
    block_sum2<kBcgBS>(rr, 0.0, part);
}

// Partials of a.b and c.d.
__global__ __launch_bounds__(kBcgBS) void k_dots2(int64_t N, const double* a, const double* b,
                                                  const double* c, const double* d, double* part)
{
    double ab = 0.0, cd = 0.0;
    BCG_ROWS(i) {
        ab += a[i] * b[i];
        cd += c[i] * d[i];
    }
    block_sum2<kBcgBS>(ab, cd, part);
}

enum BcgStep : int { BCG_INIT = 0, BCG_ALPHA = 1, BCG_W = 2, BCG_END = 3, BCG_RESTART = 4, BCG_SUMS = 5 };

// Whether the solve's loop ends, or restarts, after an iteration.
__host__ __device__ inline bool bcg_small_rho(const BcgScalars& v, double eps2) { return fabs(v.rho) < eps2 * v.r0sq; }
__host__ __device__ inline bool bcg_goes_on(const BcgScalars& v, double tol2) { return v.rr > tol2; }

// Sums nb block partial pairs in block order (one workgroup: thread k sums a
// strided subset in order, then the 256 results in order) and updates the
// scalars for the step.  The latency of its loads and of the last chain of
// additions is all its time: eight loads are in flight together, and a pair
// is read at once (2048 pairs: 6.4 us before, now 5.2).
__global__ __launch_bounds__(256) void k_bcg_fin(const double* part, int64_t nb, int step, BcgScalars* sc, double tol2,
                                                 double eps2)
{
    __shared__ double2 red[256];
    if ((step == BCG_ALPHA || step == BCG_W || step == BCG_END) && sc->stop) return;
    constexpr int K = 8;
    double a = 0.0, b = 0.0;
    for (int64_t k0 = threadIdx.x; k0 < nb; k0 += 256 * K) {
        double2 v[K];
#pragma unroll
        for (int u = 0; u < K; u++)
            v[u] = reinterpret_cast<const double2*>(part)[k0 + 256 * u < nb ? k0 + 256 * u : k0];
#pragma unroll
        for (int u = 0; u < K; u++)
            if (k0 + 256 * u < nb) {
                a += v[u].x;
                b += v[u].y;
            }
    }
    red[threadIdx.x] = make_double2(a, b);
    __syncthreads();
    if (threadIdx.x != 0) return;
    double A = 0.0, B = 0.0;
#pragma unroll 16
    for (int k = 0; k < 256; k++) { A += red[k].x; B += red[k].y; }
    switch (step) {
    case BCG_INIT:                       // r.r (= r0.r0 = r0.r), b.b; rho = alpha = w = 1
        sc->rr = A; sc->r0sq = A; sc->bb = B;
        sc->alpha = 1.0; sc->w = 1.0;
        sc->rho_old = 1.0; sc->rho = A;  // the first iteration's rho_old = rho, rho = r0.r
        sc->stop = 0;
        break;
    case BCG_ALPHA:
        sc->r0v = A;
        sc->alpha = sc->rho / A;
        break;
    case BCG_W:
        sc->tt = A; sc->ts = B;
        sc->w = A > 0.0 ? B / A : 0.0;
        break;
    case BCG_END:                        // r.r, and the next iteration's rho_old, rho
        sc->rr = A;
        sc->rho_old = sc->rho;
        sc->rho = B;
        sc->stop = !bcg_goes_on(*sc, tol2) || bcg_small_rho(*sc, eps2);
        break;
    case BCG_RESTART:                    // rho = |r0|^2 = |r|^2 (rho_old kept)
        sc->rr = A; sc->r0sq = A; sc->rho = A;
        sc->stop = 0;
        break;
    case BCG_SUMS:                       // the two sums as they are
        sc->tt = A; sc->ts = B;
        break;
    }
}

// |flow|^2 over 4 N entries and whether the velocity (first 3 N) has a NaN.
__global__ __launch_bounds__(kBcgBS) void k_flow_check(const double* flow, int64_t N, double* part)
{
    double sq = 0.0, nan = 0.0;
    BCG_ROWS(i) {
        for (int c = 0; c < 4; c++) {
            const double f = flow[c * N + i];
            sq += f * f;
            if (c < 3 && f != f) nan = 1.0;
        }
    }
    block_sum2<kBcgBS>(sq, nan, part);
}

// ============================================================================
// Per-field interface counts (batches): ranks at the field boundaries
// ============================================================================
__device__ __forceinline__ uint64_t low_mask(int b) { return b ? ((1ull << b) - 1ull) : 0ull; }

// crossing tets before tet t (t <= T): block prefix + words of the block
__device__ inline uint32_t tet_rank(int64_t t, int64_t T, const uint64_t* tbits,
                                    const uint64_t* blk_prefix, uint32_t X)
{
    if (t >= T) return X;
    uint32_t r = (uint32_t)(blk_prefix[t >> 8] >> 32);
    for (int64_t w = (t >> 8) << 2; w < (t >> 6); w++) r += __popcll(tbits[w]);
    return r + __popcll(tbits[t >> 6] & low_mask((int)(t & 63)));
}

__device__ inline uint32_t edge_rank_at(int64_t e, int64_t E, const uint64_t* ebits,
                                        const uint32_t* eprefix, uint32_t P)
{
    if (e >= E) return P;
    return eprefix[e >> 6] + (uint32_t)__popcll(ebits[e >> 6] & low_mask((int)(e & 63)));
}

// out[3f..3f+2] = (crossing points, triangles, crossing tets) of field f
__global__ void k_field_counts(int nf, const int64_t* tet_off, const int64_t* edge_off, int64_t T,
                               int64_t E, const uint64_t* tbits, const uint64_t* blk_prefix,
                               const int32_t* xtri_off, const uint64_t* ebits,
                               const uint32_t* eprefix, const uint64_t* sc, int64_t* out)
{
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nf || halted(sc)) return;
    const uint32_t X = (uint32_t)cnt_xtets(sc), F = (uint32_t)cnt_tris(sc), P = (uint32_t)cnt_points(sc);
    const uint32_t x0 = tet_rank(tet_off[f], T, tbits, blk_prefix, X);
    const uint32_t x1 = tet_rank(tet_off[f + 1], T, tbits, blk_prefix, X);
    const uint32_t f0 = x0 < X ? (uint32_t)xtri_off[x0] : F;
    const uint32_t f1 = x1 < X ? (uint32_t)xtri_off[x1] : F;
    const uint32_t p0 = edge_rank_at(edge_off[f], E, ebits, eprefix, P);
    const uint32_t p1 = edge_rank_at(edge_off[f + 1], E, ebits, eprefix, P);
    out[3 * f + 0] = p1 - p0;
    out[3 * f + 1] = f1 - f0;
    out[3 * f + 2] = x1 - x0;
}

// ============================================================================
// Kuhn grids generated on the device, numbered exactly as ft_kuhn_mesh
// ============================================================================
struct KuhnField {
    int nx, ny, nz, pad;
    double origin[3], spacing[3];
    double jitter;
    uint64_t seed;
    int64_t node_off, tet_off, edge_off;
};

__device__ __forceinline__ uint64_t mix64(uint64_t z)
{
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

__constant__ int c_kdir[7][3] = {{1,0,0},{0,1,0},{0,0,1},{1,1,0},{1,0,1},{0,1,1},{1,1,1}};
__constant__ int c_kperm[6][3] = {{0,1,2},{0,2,1},{1,0,2},{1,2,0},{2,0,1},{2,1,0}};

// Edges numbered by low node (x-major), then direction x,y,z,xy,xz,yz,xyz; a
// node has (1+I)(1+J)(1+K)-1 of them (I = not on the upper x face, ...), so the
// count before node (i,j,k) factorises over the axes.
__device__ inline int64_t kuhn_edges_before(int64_t i, int64_t j, int64_t k, int64_t X, int64_t Y,
                                            int64_t Z)
{
    auto S = [](int64_t q, int64_t Q) { return q + (q < Q - 1 ? q : Q - 1); };
    const int64_t I = i < X - 1, J = j < Y - 1;
    return (S(i, X) * S(Y, Y) * S(Z, Z) - i * Y * Z) + ((1 + I) * S(j, Y) * S(Z, Z) - j * Z) +
           ((1 + I) * (1 + J) * S(k, Z) - k);
}

__device__ inline bool kuhn_valid(int64_t i, int64_t j, int64_t k, int d, int64_t X, int64_t Y,
                                  int64_t Z)
{
    return (c_kdir[d][0] == 0 || i < X - 1) && (c_kdir[d][1] == 0 || j < Y - 1) &&
           (c_kdir[d][2] == 0 || k < Z - 1);
}

__device__ inline int32_t kuhn_edge_id(int64_t i, int64_t j, int64_t k, int d, int64_t X, int64_t Y,
                                       int64_t Z)
{
    int r = 0;
    for (int q = 0; q < d; q++) r += kuhn_valid(i, j, k, q, X, Y, Z);
    return (int32_t)(kuhn_edges_before(i, j, k, X, Y, Z) + r);
}

__global__ __launch_bounds__(kBS) void k_kuhn_nodes(KuhnField f, float* xyz)
{
    const int64_t X = f.nx, Y = f.ny, Z = f.nz;
    const int64_t a = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (a >= X * Y * Z) return;
    const int64_t i = a / (Y * Z), j = (a / Z) % Y, k = a % Z;
    const bool interior = i > 0 && i < X - 1 && j > 0 && j < Y - 1 && k > 0 && k < Z - 1;
    const int64_t ijk[3] = {i, j, k};
    float* out = xyz + 3 * (f.node_off + a);
    for (int c = 0; c < 3; c++) {
        double g = (double)ijk[c];
        if (f.jitter > 0.0 && interior) {
            const uint64_t z = mix64(f.seed + (3 * (uint64_t)a + c + 1) * 0x9E3779B97F4A7C15ULL);
            const double u = (double)(z >> 11) * 0x1.0p-53;
            g += (2.0 * u - 1.0) * f.jitter;
        }
        out[c] = (float)(f.origin[c] + g * f.spacing[c]);
    }
}

__global__ __launch_bounds__(kBS) void k_kuhn_edges(KuhnField f, int2* edges)
{
    const int64_t X = f.nx, Y = f.ny, Z = f.nz;
    const int64_t a = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (a >= X * Y * Z) return;
    const int64_t i = a / (Y * Z), j = (a / Z) % Y, k = a % Z;
    int64_t e = f.edge_off + kuhn_edges_before(i, j, k, X, Y, Z);
    for (int d = 0; d < 7; d++) {
        if (!kuhn_valid(i, j, k, d, X, Y, Z)) continue;
        const int64_t b = ((i + c_kdir[d][0]) * Y + (j + c_kdir[d][1])) * Z + (k + c_kdir[d][2]);
        edges[e++] = make_int2((int32_t)(f.node_off + a), (int32_t)(f.node_off + b));
    }
}

__global__ __launch_bounds__(kBS) void k_kuhn_tets(KuhnField f, int4* tets, int32_t* t2e)
{
    const int64_t X = f.nx, Y = f.ny, Z = f.nz;
    const int64_t CX = X - 1, CY = Y - 1, CZ = Z - 1;
    const int64_t t = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (t >= 6 * CX * CY * CZ) return;
    const int64_t cell = t / 6;
    const int p = (int)(t % 6);
    int64_t v[4][3];
    v[0][0] = cell / (CY * CZ); v[0][1] = (cell / CZ) % CY; v[0][2] = cell % CZ;
    for (int q = 1; q <= 3; q++) {
        for (int c = 0; c < 3; c++) v[q][c] = v[q - 1][c];
        v[q][c_kperm[p][q - 1]] += 1;
    }
    int32_t nd[4];
    for (int q = 0; q < 4; q++) nd[q] = (int32_t)(f.node_off + (v[q][0] * Y + v[q][1]) * Z + v[q][2]);
    tets[f.tet_off + t] = make_int4(nd[0], nd[1], nd[2], nd[3]);
    const int loc[6][2] = {{0,1},{0,2},{0,3},{1,2},{1,3},{2,3}};
    for (int q = 0; q < 6; q++) {
        const int64_t* lo = v[loc[q][0]];
        const int64_t* hi = v[loc[q][1]];
        const int dx = (int)(hi[0] - lo[0]), dy = (int)(hi[1] - lo[1]), dz = (int)(hi[2] - lo[2]);
        int d = 0;
        for (int r = 0; r < 7; r++)
            if (c_kdir[r][0] == dx && c_kdir[r][1] == dy && c_kdir[r][2] == dz) d = r;
        t2e[6 * (f.tet_off + t) + q] = (int32_t)(f.edge_off + kuhn_edge_id(lo[0], lo[1], lo[2], d, X, Y, Z));
    }
}

// Localised copies of index arrays (local -> global): mesh uploads and batch
// assembly from resident meshes.  Negative entries (slot padding) stay.
__global__ __launch_bounds__(kBS) void k_add_offset(const int32_t* src, int64_t n, int64_t add,
                                                    int32_t* dst)
{
    const int64_t i = (int64_t)blockIdx.x * kBS + threadIdx.x;
    if (i < n) dst[i] = (int32_t)(src[i] + add);
}

// Batch assembly: the concatenation of per-field pieces into one array in
// one launch.  Piece p fills dst[off[p], off[p+1]) from src[p] (element
// e - off[p]) plus add[p], or with the constant add[p] when src[p] is null;
// with keep_neg, negative source values (padding slots) are kept as they
// are.  A block copies kGatherChunk consecutive elements; it finds its first
// piece by binary search and its threads step to the next piece as they
// cross a boundary.  32-bit words: float arrays copy bit for bit (add 0).
constexpr int kGatherChunk = kBS * 8;
__global__ __launch_bounds__(kBS) void k_gather(const int32_t* const* src, const int64_t* off,
                                                const int64_t* add, int np, int keep_neg, int32_t* dst)
{
    __shared__ int p0;
    const int64_t total = off[np];
    const int64_t c0 = (int64_t)blockIdx.x * kGatherChunk;
    if (c0 >= total) return;
    if (threadIdx.x == 0) p0 = ftd::field_of(off, np, c0);
    __syncthreads();
    int p = p0;
    for (int j = 0; j < kGatherChunk / kBS; j++) {
        const int64_t e = c0 + (int64_t)j * kBS + threadIdx.x;
        if (e >= total) break;
        while (e >= off[p + 1]) p++;
        const int32_t* sp = src[p];
        if (!sp) { dst[e] = (int32_t)add[p]; continue; }
        const int32_t v = sp[e - off[p]];
        dst[e] = (keep_neg && v < 0) ? v : (int32_t)(v + add[p]);
    }
}

// ============================================================================
// Host side
// ============================================================================
struct DevBuf {
    void* p = nullptr;
    size_t cap = 0;
    template <class T> T* as() const { return static_cast<T*>(p); }
};

}  // namespace

struct FieldHost {
    float lo[3], hi[3];
    float h;                         // mean node spacing estimate
};

struct Caps {
    int64_t X = 0;   // crossing tets
    int64_t F = 0;   // triangles
    int64_t P = 0;   // crossing points
};

// A captured reinit and what it was captured for.
struct GraphState {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    double* phi = nullptr;
    double* phi_ifn = nullptr;
    ft_opts opts{};
    uint64_t layout = 0;
    Caps caps;
    std::vector<void*> bufs;         // device buffers the graph's kernels address
    int64_t captures = 0, launches = 0;
};

struct ft_ctx {
    int device = 0;
    int cu_count = 256;              // compute units of the device
    hipStream_t stream = nullptr;
    // A second stream for the stages the query does not read (the interface's
    // point-to-triangle lists and areas) and the query's tile schedule: they
    // run beside the index build.  side_fork/side_join order it against the
    // calling stream; side_open: forked and not joined yet.
    hipStream_t side = nullptr;
    hipEvent_t side_fork_ev = nullptr, side_join_ev = nullptr;
    bool side_open = false;
    // fields and mesh (field k: nodes [node_off[k], node_off[k+1]), ...)
    int nf = 0;
    std::vector<int64_t> node_off, tet_off, edge_off, slot_off;
    std::vector<FieldHost> fh;
    int64_t N = 0, T = 0, E = 0, n_slots = 0;
    uint64_t layout_gen = 0;         // bumped whenever the fields change
    bool has_conn = false;
    float h_est = 0.0f;
    DevBuf xyz, tets, edges, t2e, perm, sx, sy, sz, tile_field;
    DevBuf tile_sched;               // per query tile: class, launch order, class scan
    DevBuf deep_part;                // the parts' keys of the split tiles
    DevBuf gather_tab;               // piece tables of the batch assembly (ft_set_batch_meshes)
    // A batch of resident meshes reads their tets, t2e and edges in place
    // (virt): field_tab holds the per-field pointers, field_meshes keeps the
    // meshes alive while the batch refers to them.  Operations that need the
    // concatenated arrays copy them once (materialize_conn).
    bool virt = false;
    DevBuf field_tab;
    std::vector<std::shared_ptr<ft_ctx>> field_meshes;
    DevBuf d_node_off, d_tet_off, d_edge_off, d_slot_off;
    // per reinit
    DevBuf phi_tmp, phi_ifn_tmp;
    DevBuf sbits, retain, tbits, blk, xtet, xtri_off, xedges, ebits, eprefix;
    DevBuf ifp, ifp2e, tris, tri_norm, if_elems, p2t_off, p2t_cursor, p2t, ifp_area;
    DevBuf nearest, fcounts, fclamp;
    // normals: node -> tets lists (per field layout), tet gradients, node normals
    DevBuf n2t_off, n2t_ids, grad_t, normals, phi_ifn_int;
    DevBuf gsplit, kmesh, k_if;      // curvature: unit-normal components, node and point curvature
    DevBuf st_cnt, st_off, st_ids;   // surface tension: node -> crossing-point terms
    DevBuf st_f;                     // surface tension: device copy of host force arrays
    // advection: sliced-ELL pattern and mass matrix (per layout), the
    // Crank-Nicolson matrix, BiCGSTAB vectors, block partials and scalars
    DevBuf fem_len, fem_w, fem_soff, fem_cols, fem_nd, fem_diag, fem_dmask, fem_m, fem_l, fem_flag, fem_map;
    DevBuf bcg_vec, bcg_part, bcg_sc, adv_phi, adv_flow, adv_vel3, fem_csr_off;
    uint64_t fem_layout = ~0ull;
    int64_t fem_nnz = 0;             // ELL entries with padding
    int fem_stride = 1;              // LDS doubles per row accumulator (longest row, odd)
    void* h_bcg = nullptr;           // pinned mirrors of the solver scalars: one, and one per iteration in flight
    hipEvent_t bcg_ev[kBcgAhead] = {};
    const double* last_phi = nullptr;   // device phi of the last reinit (blended)
    uint64_t n2t_layout = ~0ull;
    bool tets_twice = false;         // a tet names a node twice (found with the node -> tets lists)
    bool have_normals = false;
    // index
    DevBuf bin_count, bin_prefix;    // the node sort's bins (mesh set-up)
    DevBuf bbits, bprefix, pcode, place, prec, titem, trec, pidx;
    DevBuf leaf_cnt, leaf_bin, nfirst, nitem, naxis, stats;
    DevBuf d_grids, d_cnt_off, roots;
    uint64_t idx_layout = ~0ull;     // layout, bin scale and reach the grids were made for
    float idx_bin_scale = 0.0f, idx_reach = 0.0f;
    int64_t idx_G = 0;               // bins over all fields (a multiple of 64)
    int64_t idx_words[5] = {0, 0, 0, 0, 0};   // blocks of 64^k bins over all fields
    int idx_top = 1;                 // highest level that holds a field's root
    GraphState graph;
    // capacities for the next eager call on the same fields and mode
    Caps spec_caps;
    uint64_t spec_layout = ~0ull;
    int spec_mode = -1;
    int64_t spec_hits = 0;
    // scan scratch and small scalars
    DevBuf scan_bsum, scalars;
    DevBuf scan_side;                // scan scratch of the side stream
    uint64_t* h_scalars = nullptr;   // pinned mirror
    ft_counts last{};
    std::vector<ft_counts> field_counts;
    std::vector<uint64_t> batch_meshes;  // serials of the resident meshes of the current batch
    bool have_interface = false;
    bool have_nearest = false;
    // phase timing (ft_set_timing): events at the phase boundaries of a reinit
    bool timing = false;
    hipEvent_t ev[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
    // host <-> device staging of large host arrays: two pinned chunks
    void* stage[2] = {nullptr, nullptr};
    hipEvent_t stage_ev[2] = {nullptr, nullptr};
    double phase_ms[4] = {0, 0, 0, 0};
    int64_t timed_calls = 0;
};

namespace {

void drop_graph(ft_ctx* c);
int materialize_conn(ft_ctx* h);

std::vector<DevBuf*> all_buffers(ft_ctx* h)
{
    return {&h->xyz, &h->tets, &h->edges, &h->t2e, &h->perm, &h->sx, &h->sy, &h->sz,
            &h->tile_field, &h->tile_sched, &h->gather_tab, &h->field_tab, &h->d_node_off, &h->d_tet_off, &h->d_edge_off, &h->d_slot_off,
            &h->fcounts, &h->fclamp, &h->d_grids, &h->d_cnt_off, &h->roots,
            &h->phi_tmp, &h->phi_ifn_tmp, &h->sbits, &h->retain, &h->tbits, &h->blk,
            &h->xtet, &h->xtri_off, &h->xedges, &h->ebits, &h->eprefix, &h->ifp,
            &h->ifp2e, &h->tris, &h->tri_norm, &h->if_elems, &h->p2t_off,
            &h->p2t_cursor, &h->p2t, &h->ifp_area, &h->nearest, &h->bin_count,
            &h->bin_prefix, &h->bbits, &h->bprefix, &h->pcode, &h->place, &h->prec, &h->titem, &h->trec,
            &h->pidx, &h->leaf_cnt, &h->leaf_bin, &h->nfirst, &h->nitem, &h->naxis, &h->stats, &h->scan_bsum, &h->scan_side, &h->deep_part, &h->scalars,
            &h->n2t_off, &h->n2t_ids, &h->grad_t, &h->normals, &h->phi_ifn_int,
            &h->gsplit, &h->kmesh, &h->k_if, &h->st_cnt, &h->st_off, &h->st_ids, &h->st_f,
            &h->fem_len, &h->fem_w, &h->fem_soff, &h->fem_cols, &h->fem_nd, &h->fem_diag, &h->fem_dmask, &h->fem_m, &h->fem_l, &h->fem_flag, &h->fem_map,
            &h->bcg_vec, &h->bcg_part, &h->bcg_sc, &h->adv_phi, &h->adv_flow, &h->adv_vel3, &h->fem_csr_off};
}

std::vector<void*> buffer_addresses(ft_ctx* c)
{
    std::vector<void*> a;
    for (DevBuf* b : all_buffers(c)) a.push_back(b->p);
    return a;
}

// Workspace of an allocation-free call (ft_reinit_device_noalloc): while it
// is set on the calling thread, ensure() hands out consecutive pieces of it
// instead of allocating, and release() drops buffers without freeing.
struct Arena {
    char* base = nullptr;
    size_t size = 0, used = 0;
};
thread_local Arena* t_arena = nullptr;

int ensure(DevBuf& b, size_t bytes)
{
    if (bytes == 0) bytes = 16;
    if (bytes <= b.cap) return FT_OK;
    if (t_arena) {
        const size_t want = (bytes + 255) & ~(size_t)255;
        if (t_arena->used + want > t_arena->size)
            return ft::set_error(FT_ERR_BUDGET,
                                 "the workspace of this reinit exceeds the %zu-byte scratch of "
                                 "ft_reinit_device_noalloc (%zu bytes taken, %zu more asked); use "
                                 "ft_reinit_device", t_arena->size, t_arena->used, want);
        b.p = t_arena->base + t_arena->used;
        b.cap = want;
        t_arena->used += want;
        return FT_OK;
    }
    if (b.p) (void)hipFree(b.p);
    b.p = nullptr;
    b.cap = 0;
    size_t want = bytes + bytes / 8;
    want = (want + 255) & ~(size_t)255;
    hipError_t e = hipMalloc(&b.p, want);
    if (e != hipSuccess) {
        b.p = nullptr;
        return ft::set_error(FT_ERR_NOMEM, "hipMalloc(%zu) failed: %s", want, hipGetErrorString(e));
    }
    b.cap = want;
    return FT_OK;
}

// Whether ensure(b, bytes) would have the memory.
bool has_room(const DevBuf& b, size_t bytes)
{
    return !t_arena || bytes <= b.cap || t_arena->used + ((bytes + 255) & ~(size_t)255) <= t_arena->size;
}

void release(DevBuf& b)
{
    if (b.p && !t_arena) (void)hipFree(b.p);
    b.p = nullptr;
    b.cap = 0;
}

template <class T>
int fill(hipStream_t s, T* p, int64_t n, T v)
{
    if (n <= 0) return FT_OK;
    hipLaunchKernelGGL(k_fill<T>, dim3(grid1d(n)), dim3(kBS), 0, s, p, n, v);
    FT_HIP(hipGetLastError());
    return FT_OK;
}

int set_words(hipStream_t s, const WordRanges& r)
{
    if (r.n == 0) return FT_OK;
    hipLaunchKernelGGL(k_set_words, dim3(grid1d(r.total())), dim3(kBS), 0, s, r);
    FT_HIP(hipGetLastError());
    return FT_OK;
}

// Exclusive scan of n elements; the total lands in *d_total (device).
// ws: the block-sum scratch (default: the handle's; each stream needs its own).
template <class TI, class TO, class Ld>
int scan(ft_ctx* c, hipStream_t s, const TI* in, TO* out, int64_t n, TO* d_total, Ld ld, DevBuf* ws = nullptr)
{
    if (n <= kScanOne) {
        hipLaunchKernelGGL((k_scan_one<TI, TO, Ld>), dim3(1), dim3(1024), 0, s, in, out, n, d_total, ld);
        FT_HIP(hipGetLastError());
        return FT_OK;
    }
    DevBuf& w = ws ? *ws : c->scan_bsum;
    const int64_t nb = (n + kScanTile - 1) / kScanTile;
    FT_TRY(ensure(w, sizeof(TO) * (size_t)nb));
    TO* bs = w.as<TO>();
    hipLaunchKernelGGL((k_scan_reduce<TI, TO, Ld>), dim3((unsigned)nb), dim3(kBS), 0, s, in, n, bs, ld);
    hipLaunchKernelGGL(k_scan_top<TO>, dim3(1), dim3(1024), 0, s, bs, nb, d_total);
    hipLaunchKernelGGL((k_scan_down<TI, TO, Ld>), dim3((unsigned)nb), dim3(kBS), 0, s, in, out, n, bs, ld);
    FT_HIP(hipGetLastError());
    return FT_OK;
}

// Uniform cubic grid over a field's box with edge >= `edge` and at most
// 2^max_lg bins per axis; *lg receives log2 of the Morton side.
// reach: a power of two (far_reach); the unit of the scaled coordinates is at least this.
Grid make_grid(const FieldHost& f, float edge, int max_lg, int* lg_out, float reach = 0.0f)
{
    Grid g{};
    float ext_max = 0.0f;
    for (int k = 0; k < 3; k++) ext_max = std::max(ext_max, f.hi[k] - f.lo[k]);
    float b = std::max(edge, ext_max / (float)(1 << max_lg) * 1.0001f);
    if (!(b > 0.0f)) b = 1.0f;
    int lg = 0;
    for (int k = 0; k < 3; k++) {
        int d = (int)std::ceil((f.hi[k] - f.lo[k]) / b);
        d = std::max(1, std::min(d, 1 << max_lg));
        g.dim[k] = d;
        g.lo[k] = f.lo[k];
        while ((1 << lg) < d) lg++;
    }
    g.inv_b = 1.0f / b;
    g.h = f.h;
    // scaled coordinates: about the box's middle, in units of a power of two
    // of at least twice its longest side (scaling rounds nothing; the field
    // and what lies within half a side of it stay within one unit).  A box
    // without a finite size (a node that is not finite, or sides beyond
    // FLT_MAX): about 0, in the largest unit, in which every finite coordinate
    // stays below 4; the units' reciprocal is a normal number.
    const bool sized = ext_max <= FLT_MAX;
    int ex = 0;
    (void)std::frexp(sized ? std::max(std::max(ext_max, 0.25f * reach), 1e-30f) : FLT_MAX, &ex);   // ext_max < 2^ex
    for (int k = 0; k < 3; k++) g.org[k] = sized ? f.lo[k] + 0.5f * (f.hi[k] - f.lo[k]) : 0.0f;
    g.inv_s = std::ldexp(1.0f, -std::min(ex + 1, 126));
    g.root_lv = std::max(1, (lg + 1) / 2);
    *lg_out = lg;
    return g;
}

int field_bits(int nf)
{
    int b = 0;
    while ((1 << b) < nf) b++;
    return b;
}

int check_launch() { FT_HIP(hipGetLastError()); return FT_OK; }

// Copies `count` u64 device scalars (ctx->scalars) to the host and waits.
int read_scalars(ft_ctx* c, hipStream_t s, int count)
{
    FT_HIP(hipMemcpyAsync(c->h_scalars, c->scalars.p, sizeof(uint64_t) * count, hipMemcpyDeviceToHost, s));
    FT_HIP(hipStreamSynchronize(s));
    return FT_OK;
}

int check_handle(ft_handle h)
{
    if (!h) return ft::set_error(FT_ERR_ARG, "null handle");
    FT_HIP(hipSetDevice(h->device));
    return FT_OK;
}

// ---- Staged host <-> device copies -----------------------------------------
// A pageable copy runs at 17 GB/s (to host) to 30 GB/s (to device) on this
// platform, a pinned one at about 56 GB/s both ways.  Large host arrays go
// through two pinned chunks instead: host threads copy one chunk between
// the caller's array and pinned memory while the DMA engine moves the other.
constexpr size_t kStageChunk = size_t(32) << 20;
constexpr int kStageThreads = 4;
constexpr size_t kStageMin = size_t(8) << 20;          // smaller: one plain copy

void par_memcpy(void* dst, const void* src, size_t n)
{
    if (n < (size_t(4) << 20)) { std::memcpy(dst, src, n); return; }
    const size_t part = ((n + kStageThreads - 1) / kStageThreads + 63) & ~size_t(63);
    std::thread th[kStageThreads - 1];
    int started = 0;
    try {
        for (int t = 1; t < kStageThreads; t++) {
            const size_t lo = std::min(n, part * t), hi = std::min(n, part * (t + 1));
            if (lo >= hi) break;
            th[t - 1] = std::thread([=] { std::memcpy((char*)dst + lo, (const char*)src + lo, hi - lo); });
            started = t;
        }
    } catch (...) {                                     // no thread: copy the rest here
        const size_t lo = std::min(n, part * (started + 1));
        std::memcpy((char*)dst + lo, (const char*)src + lo, n - lo);
    }
    std::memcpy(dst, src, std::min(n, part));
    for (int t = 0; t < started; t++) th[t].join();
}

int stage_setup(ft_ctx* h)
{
    for (int k = 0; k < 2; k++) {
        if (!h->stage[k]) FT_HIP(hipHostMalloc(&h->stage[k], kStageChunk, hipHostMallocDefault));
        if (!h->stage_ev[k]) FT_HIP(hipEventCreateWithFlags(&h->stage_ev[k], hipEventDisableTiming));
    }
    return FT_OK;
}

// Host to device, enqueued on s; returns once the host array may be reused.
int copy_h2d(ft_ctx* h, void* dst, const void* src, size_t bytes, hipStream_t s)
{
    if (bytes < kStageMin) {
        if (bytes) FT_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s));
        FT_HIP(hipStreamSynchronize(s));
        return FT_OK;
    }
    FT_TRY(stage_setup(h));
    size_t off = 0;
    for (int k = 0; off < bytes; k++, off += kStageChunk) {
        const int b = k & 1;
        const size_t len = std::min(kStageChunk, bytes - off);
        if (k >= 2) FT_HIP(hipEventSynchronize(h->stage_ev[b]));   // chunk k-2 has left this buffer
        par_memcpy(h->stage[b], (const char*)src + off, len);
        FT_HIP(hipMemcpyAsync((char*)dst + off, h->stage[b], len, hipMemcpyHostToDevice, s));
        FT_HIP(hipEventRecord(h->stage_ev[b], s));
    }
    FT_HIP(hipStreamSynchronize(s));
    return FT_OK;
}

// Device to host after the work already on s, for a list of (host, device,
// bytes) segments moved as one sequence of chunks.
struct D2H {
    void* host;
    const void* dev;
    size_t bytes;
};
int copy_d2h(ft_ctx* h, const std::vector<D2H>& segs, hipStream_t s)
{
    size_t total = 0;
    for (const D2H& g : segs) total += g.bytes;
    if (total < kStageMin) {
        for (const D2H& g : segs)
            if (g.bytes) FT_HIP(hipMemcpyAsync(g.host, g.dev, g.bytes, hipMemcpyDeviceToHost, s));
        FT_HIP(hipStreamSynchronize(s));
        return FT_OK;
    }
    FT_TRY(stage_setup(h));
    struct Chunk { char* host; const char* dev; size_t len; };
    std::vector<Chunk> ch;
    for (const D2H& g : segs)
        for (size_t off = 0; off < g.bytes; off += kStageChunk)
            ch.push_back({(char*)g.host + off, (const char*)g.dev + off, std::min(kStageChunk, g.bytes - off)});
    for (size_t k = 0; k < ch.size() && k < 2; k++) {
        FT_HIP(hipMemcpyAsync(h->stage[k], ch[k].dev, ch[k].len, hipMemcpyDeviceToHost, s));
        FT_HIP(hipEventRecord(h->stage_ev[k], s));
    }
    for (size_t k = 0; k < ch.size(); k++) {
        const int b = (int)(k & 1);
        FT_HIP(hipEventSynchronize(h->stage_ev[b]));
        par_memcpy(ch[k].host, h->stage[b], ch[k].len);
        if (k + 2 < ch.size()) {
            FT_HIP(hipMemcpyAsync(h->stage[b], ch[k + 2].dev, ch[k + 2].len, hipMemcpyDeviceToHost, s));
            FT_HIP(hipEventRecord(h->stage_ev[b], s));
        }
    }
    return FT_OK;
}


// Field layout: offsets on host and device, slot layout (each field padded to
// whole waves).
int set_fields(ft_ctx* c, int nf, const int64_t* node_off, const int64_t* tet_off,
               const int64_t* edge_off)
{
    c->batch_meshes.clear();
    c->virt = false;
    c->field_meshes.clear();
    c->layout_gen++;
    c->nf = nf;
    c->node_off.assign(node_off, node_off + nf + 1);
    c->tet_off.assign(tet_off, tet_off + nf + 1);
    c->edge_off.assign(edge_off, edge_off + nf + 1);
    c->slot_off.assign(nf + 1, 0);
    c->N = node_off[nf];
    c->T = tet_off[nf];
    c->E = edge_off[nf];
    c->n_slots = 0;                  // set with the node sort (set_slots)
    c->fh.assign(nf, FieldHost{});
    c->field_counts.assign(nf, ft_counts{});
    const size_t ob = sizeof(int64_t) * (nf + 1);
    FT_TRY(ensure(c->d_node_off, ob));
    FT_TRY(ensure(c->d_tet_off, ob));
    FT_TRY(ensure(c->d_edge_off, ob));
    FT_TRY(ensure(c->d_slot_off, ob));
    FT_HIP(hipMemcpyAsync(c->d_node_off.p, c->node_off.data(), ob, hipMemcpyHostToDevice, c->stream));
    FT_HIP(hipMemcpyAsync(c->d_tet_off.p, c->tet_off.data(), ob, hipMemcpyHostToDevice, c->stream));
    FT_HIP(hipMemcpyAsync(c->d_edge_off.p, c->edge_off.data(), ob, hipMemcpyHostToDevice, c->stream));
    FT_HIP(hipStreamSynchronize(c->stream));
    return FT_OK;
}

// Query slots of each field (multiples of 64).
int set_slots(ft_ctx* c, const std::vector<int64_t>& slots)
{
    for (int k = 0; k < c->nf; k++) c->slot_off[k + 1] = c->slot_off[k] + slots[k];
    c->n_slots = c->slot_off[c->nf];
    const size_t n = (size_t)std::max<int64_t>(1, c->n_slots);
    FT_TRY(ensure(c->perm, sizeof(int32_t) * n));
    FT_TRY(ensure(c->sx, sizeof(float) * n));
    FT_TRY(ensure(c->sy, sizeof(float) * n));
    FT_TRY(ensure(c->sz, sizeof(float) * n));
    FT_TRY(ensure(c->tile_field, sizeof(int32_t) * std::max<size_t>(1, n / 64)));
    FT_TRY(ensure(c->tile_sched, 4 * sizeof(int32_t) * std::max<size_t>(1, n / 64)));
    // (both callers wait for the stream before they return)
    FT_HIP(hipMemcpyAsync(c->d_slot_off.p, c->slot_off.data(), sizeof(int64_t) * (c->nf + 1), hipMemcpyHostToDevice,
                          c->stream));
    return FT_OK;
}

void finish_field_box(FieldHost& f, int64_t n)
{
    if (n == 0) for (int k = 0; k < 3; k++) { f.lo[k] = 0; f.hi[k] = 1; }
    double vol = 1.0, ext_max = 0.0;
    for (int k = 0; k < 3; k++) ext_max = std::max(ext_max, (double)f.hi[k] - f.lo[k]);
    if (!(ext_max > 0.0)) ext_max = 1.0;
    for (int k = 0; k < 3; k++) vol *= std::max((double)f.hi[k] - f.lo[k], ext_max * 1e-3);
    f.h = (float)std::cbrt(vol / (double)std::max<int64_t>(1, n));
}

// Field boxes from host coordinates.
void boxes_from_host(ft_ctx* c, const float* xyz)
{
    for (int k = 0; k < c->nf; k++) {
        FieldHost& f = c->fh[k];
        for (int q = 0; q < 3; q++) { f.lo[q] = FLT_MAX; f.hi[q] = -FLT_MAX; }
        for (int64_t i = c->node_off[k]; i < c->node_off[k + 1]; i++)
            for (int q = 0; q < 3; q++) {
                f.lo[q] = std::min(f.lo[q], xyz[3 * i + q]);
                f.hi[q] = std::max(f.hi[q], xyz[3 * i + q]);
            }
        finish_field_box(f, c->node_off[k + 1] - c->node_off[k]);
    }
    c->h_est = c->nf ? c->fh[0].h : 0.0f;
}

// Grid of the node sort.  A query wave takes 64 consecutive slots, so the
// tiles are compact only if the bins follow the nodes.  When a field's node
// count and box fit a structured grid -- n = nx ny nz nodes with nx - 1,
// ny - 1, nz - 1 spacings s along the box's edges, as a box mesher's (or
// the Kuhn generator's) grid, jittered by less than s / 2 -- the bins are
// kf s wide and start s / 2 before the box: every bin then holds the
// kf^3 nodes of one block (kf = 1 or 2), and *cpb consecutive bins along the
// Morton curve an aligned 4 x 4 x 4 block of nodes, which gets a tile of its
// own: *tiles in all.  Packed without gaps, a grid whose sides are no
// multiples of 4 has its blocks cut by the tiles, and a tile that holds the
// end of one octant and the start of the next spans half the field (127^3:
// the last 2% of the tiles took as long as the rest).  Grids whose
// blocks would be emptier than kBlockFill keep the packed order (*cpb = 0),
// as does any other field, on a grid of about one node per bin.  The order
// only affects speed: each node's result is the same in any slot.
// Blocks against packed slots, a reinit to the triangles: 33^3 (0.77 full) 272
// and 342 us, 65^3 (0.89) 380 and 467, 129 x 33 x 9 (0.67) 356 and 537; 17^3
// (0.61) and 25^3 (0.72) the same within 2 %, as are 9^3, 13^3, 129 x 129 x 5 and
// 900 x 9 x 9 (0.42 to 0.60), where blocks would only take more slots.  37^3
// (0.79) loses 2 %, to the points 9 %.
constexpr double kBlockFill = 0.6;
Grid node_sort_grid(const FieldHost& f, int64_t n, int max_lg, int* lg_out, int* cpb, int64_t* tiles)
{
    *cpb = 0;
    *tiles = (n + 63) / 64;
    const Grid fallback = make_grid(f, f.h, max_lg, lg_out);
    double ext[3], ext_max = 0.0;
    for (int k = 0; k < 3; k++) {
        ext[k] = (double)f.hi[k] - f.lo[k];
        if (!(ext[k] >= 0.0)) return fallback;
        ext_max = std::max(ext_max, ext[k]);
    }
    if (n < 8 || !(ext_max > 0.0)) return fallback;
    // prod_k (ext_k / s + 1) decreases in s: bisection for the s that gives n
    auto count = [&](double s) {
        double p = 1.0;
        for (int k = 0; k < 3; k++) p *= ext[k] / s + 1.0;
        return p;
    };
    double lo_s = ext_max / (double)n, hi_s = ext_max;   // count(lo_s) > n >= 8 >= count(hi_s)
    if (!(count(hi_s) <= (double)n)) return fallback;
    for (int it = 0; it < 200; it++) {
        const double mid = 0.5 * (lo_s + hi_s);
        (count(mid) > (double)n ? lo_s : hi_s) = mid;
    }
    const double s0 = 0.5 * (lo_s + hi_s);
    int64_t nk[3], prod = 1, cells = 1;
    double s_sum = 0.0;
    int s_cnt = 0;
    for (int k = 0; k < 3; k++) {
        const double q = ext[k] / s0 + 1.0;
        nk[k] = std::llround(q);
        if (nk[k] < 1 || std::fabs(q - (double)nk[k]) > 0.05) return fallback;
        prod *= nk[k];
        cells = std::max(cells, nk[k]);
        if (nk[k] > 1) { s_sum += ext[k] / (double)(nk[k] - 1); s_cnt++; }
    }
    if (prod != n || s_cnt == 0) return fallback;
    const double s = s_sum / s_cnt;
    for (int k = 0; k < 3; k++)
        if (nk[k] > 1 && std::fabs(ext[k] / (double)(nk[k] - 1) - s) > 1e-4 * s) return fallback;
    const int64_t kf = (cells + (1ll << max_lg) - 1) >> max_lg;   // spacings per bin
    if (kf > 2) return fallback;                                   // blocks would not be 4 x 4 x 4
    Grid g{};
    int lg = 0;
    for (int k = 0; k < 3; k++) {
        g.lo[k] = (float)((double)f.lo[k] - 0.5 * s);
        // node i of the axis lands in bin floor((i + 1/2) / kf)
        g.dim[k] = (int)(((nk[k] - 1) * 2 + 1) / (2 * kf)) + 1;
        while ((1 << lg) < g.dim[k]) lg++;
    }
    g.inv_b = (float)(1.0 / ((double)kf * s));
    g.h = f.h;
    *lg_out = lg;
    int64_t blocks = 1;
    for (int k = 0; k < 3; k++) blocks *= (nk[k] + 3) / 4;
    const int block_bins = kf == 1 ? 64 : 8;
    if ((double)n >= kBlockFill * 64.0 * (double)blocks && ((int64_t)1 << (3 * lg)) >= block_bins) {
        *cpb = block_bins;
        *tiles = blocks;
    }
    return g;
}

// Morton order of each field's nodes into the query slots (device xyz):
// one counting sort per field on node_sort_grid.  blocks: a tile per block of
// a structured grid; a field that only looked like one (a block of more than
// 64 nodes, or an empty one) sends the whole handle back to the packed order.
int sort_nodes(ft_ctx* c, bool blocks = true)
{
    const int nf = c->nf;
    std::vector<Grid> grids(nf);
    std::vector<int> lgs(nf, 0), cpb(nf, 0);
    std::vector<int64_t> slots(nf, 0);
    int64_t max_bins = 1, max_blocks = 0, max_n = 1;   // of a field
    for (int k = 0; k < nf; k++) {
        const int64_t n = c->node_off[k + 1] - c->node_off[k];
        int64_t tiles = 0;
        if (n > 0) grids[k] = node_sort_grid(c->fh[k], n, kMaxBinsLog2PerAxis, &lgs[k], &cpb[k], &tiles);
        if (!blocks && cpb[k]) {
            cpb[k] = 0;
            tiles = (n + 63) / 64;
        }
        slots[k] = 64 * tiles;
        const int64_t bins = (int64_t)1 << (3 * lgs[k]);
        max_bins = std::max(max_bins, bins);
        max_blocks = std::max(max_blocks, cpb[k] ? bins / cpb[k] : 0);
        max_n = std::max(max_n, n);
    }
    FT_TRY(set_slots(c, slots));
    hipStream_t s = c->stream;
    if (c->N == 0) {
        FT_HIP(hipStreamSynchronize(s));
        return FT_OK;
    }
    FT_TRY(ensure(c->bin_count, sizeof(uint32_t) * max_bins));
    FT_TRY(ensure(c->bin_prefix, sizeof(uint32_t) * (max_bins + max_blocks)));
    FT_TRY(ensure(c->pcode, sizeof(uint32_t) * max_n));
    // raised by the kernels, in the pinned mirror, so that nothing is read back
    unsigned long long* misfit = reinterpret_cast<unsigned long long*>(c->h_scalars) + S_P2T;
    *misfit = 0ull;
    WordRanges clr;                                    // once: a field leaves its bins' counts at zero
    clr.add(c->perm.p, c->n_slots, ~0u);
    clr.add(c->bin_count.p, max_bins, 0u);
    FT_TRY(set_words(s, clr));
    for (int k = 0; k < nf; k++) {
        const int64_t n = c->node_off[k + 1] - c->node_off[k];
        if (n == 0) continue;
        const Grid& g = grids[k];
        const int64_t G = (int64_t)1 << (3 * lgs[k]);
        const int64_t nb = cpb[k] ? G / cpb[k] : 0;   // blocks
        uint32_t* cnt = c->bin_count.as<uint32_t>();
        uint32_t* off = c->bin_prefix.as<uint32_t>();
        uint32_t* btile = off + G;                     // per block
        uint32_t* total = reinterpret_cast<uint32_t*>(c->scalars.as<uint64_t>() + S_BINS);
        const float* xk = c->xyz.as<float>() + 3 * c->node_off[k];
        const int64_t sb = c->slot_off[k];
        hipLaunchKernelGGL(k_node_bin, dim3(grid1d(n)), dim3(kBS), 0, s, xk, n, g, c->pcode.as<uint32_t>(), cnt);
        if (cpb[k]) {
            FT_TRY(scan<uint32_t, uint32_t>(c, s, cnt, off, G, total, LoadBlocks{cpb[k], btile}));
            FT_TRY(scan<uint32_t, uint32_t>(c, s, btile, btile, nb, total, LoadSame{}));
        } else {
            FT_TRY(scan<uint32_t, uint32_t>(c, s, cnt, off, G, total, LoadSame{}));
        }
        hipLaunchKernelGGL(k_node_scatter, dim3(grid1d(n)), dim3(kBS), 0, s, xk, n, c->node_off[k],
                           c->pcode.as<uint32_t>(), cnt, off, cpb[k], btile, slots[k], misfit,
                           c->perm.as<int32_t>() + sb, c->sx.as<float>() + sb, c->sy.as<float>() + sb,
                           c->sz.as<float>() + sb);
    }
    hipLaunchKernelGGL(k_pad_slots, dim3(grid1d(c->n_slots)), dim3(kBS), 0, s, c->n_slots, nf,
                       c->d_slot_off.as<int64_t>(), c->perm.as<int32_t>(), c->sx.as<float>(),
                       c->sy.as<float>(), c->sz.as<float>(), c->tile_field.as<int32_t>(), misfit);
    FT_TRY(check_launch());
    FT_HIP(hipStreamSynchronize(s));
    if (*(volatile unsigned long long*)misfit) {
        if (!blocks) return ft::set_error(FT_ERR_INTERNAL, "node sort: more nodes than slots");
        return sort_nodes(c, false);
    }
    return FT_OK;
}

// ----------------------------------------------------------------------------
// One reinit: stage buffers, the kernel sequence, and the readback
// ----------------------------------------------------------------------------
// Buffer capacities of one reinit, in elements.  An eager reinit sizes them
// to the exact stage totals it reads back between stages.  A captured graph
// fixes them when it is captured; the device then raises S_CAP when a total
// outgrows them, every later kernel does nothing, and the host captures again
// with more room (phi is only written by the last kernel, so nothing is lost).
// Default bin edge, in node spacings, per distance mode (0 points, 1
// triangles).  A bin's primitives form one leaf.  Points are cheap to test and
// their least-squares-plane box tightens with more points, so their
// optimum is larger.  A whole reinit (64 spheres), triangles at 1.0 / 1.25 / 1.5 /
// 2.0 / 2.5: 256^3 7.33 / 7.41 / 7.48 / 7.41 / 8.26 ms, 128^3 1.33 / 1.37 / 1.25 /
// 1.29 / 1.39, 64^3 0.49 / 0.49 / 0.50 / 0.51 / 0.52; points at 1.5 / 2.0 / 2.5 / 3.0:
// 256^3 4.59 / 4.14 / 4.14 / 4.31, 128^3 0.86 / 0.82 / 0.82 / 0.83.
constexpr float kDefaultBinScale[2] = {2.0f, 1.25f};

// For given points that may lie far outside the mesh: a bound on the distance
// of every node of the field to its nearest point, as a power of two, if that
// is more than a unit of make_grid; else 0 (the first point inside the box, or
// near it, says so).  The search cuts distances along an axis at one unit: with
// all points beyond it every box would be admitted (48^3 nodes, 6000 points on a
// sphere 7.5 sides off: 846 us, and 280 with units of that size).
float far_reach(const FieldHost& f, const float* p, int64_t n)
{
    double c[3], ext_max = 0.0, half2 = 0.0, near2 = INFINITY;
    for (int k = 0; k < 3; k++) {
        const double e = (double)f.hi[k] - f.lo[k];
        c[k] = 0.5 * ((double)f.lo[k] + f.hi[k]);
        ext_max = std::max(ext_max, e);
        half2 += 0.25 * e * e;
    }
    const double near_enough = 2.0 * ext_max - std::sqrt(half2);
    if (!(near_enough < FLT_MAX)) return 0.0f;
    for (int64_t j = 0; j < n; j++) {
        double d2 = 0.0;
        for (int k = 0; k < 3; k++) d2 += (p[3 * j + k] - c[k]) * (p[3 * j + k] - c[k]);
        near2 = d2 < near2 ? d2 : near2;                             // (not for a NaN)
        if (near2 <= near_enough * near_enough) return 0.0f;
    }
    const double reach = std::sqrt(near2) + std::sqrt(half2);
    if (!(reach < 0.25 * FLT_MAX)) return 0.0f;
    int e = 0;
    (void)std::frexp((float)reach * (1.0f + 0x1.0p-20f), &e);
    return std::ldexp(1.0f, e);
}

// Per-field bin grids of the index for one bin_scale (0: the mode's default)
// and reach, on the device; cached per field layout.
int index_setup(ft_ctx* c, hipStream_t s, float bin_scale, int mode, float reach = 0.0f)
{
    const float bs = bin_scale > 0.0f ? bin_scale : kDefaultBinScale[mode];
    if (c->idx_layout == c->layout_gen && c->idx_bin_scale == bs && c->idx_reach == reach) return FT_OK;
    const int nf = c->nf;
    const int fb = field_bits(nf);
    // bins of all fields together stay near 2^30
    const int max_lg = std::min(kMaxBinsLog2PerAxis, (30 - fb) / 3);
    std::vector<Grid> grids(nf);
    std::vector<int64_t> cnt_off(nf + 1, 0);
    int64_t words[kLevels] = {0, 0, 0, 0, 0};
    int top = 1;
    for (int k = 0; k < nf; k++) {
        int lg = 0;
        grids[k] = make_grid(c->fh[k], bs * c->fh[k].h, max_lg, &lg, reach);
        top = std::max(top, grids[k].root_lv);
        const int64_t bins = (int64_t)1 << (3 * lg);
        cnt_off[k + 1] = cnt_off[k] + std::max<int64_t>(64, bins);   // whole bitmap words
        for (int q = 1; q < kLevels; q++) words[q] += std::max<int64_t>(1, bins >> (6 * q));
    }
    const int64_t G = cnt_off[nf];
    if (G > ((int64_t)1 << 32))
        return ft::set_error(FT_ERR_ARG, "index: %lld bins exceed 2^32; raise bin_scale", (long long)G);
    FT_TRY(ensure(c->d_grids, sizeof(Grid) * nf));
    FT_TRY(ensure(c->d_cnt_off, sizeof(int64_t) * (nf + 1)));
    FT_HIP(hipMemcpyAsync(c->d_grids.p, grids.data(), sizeof(Grid) * nf, hipMemcpyHostToDevice, s));
    FT_HIP(hipMemcpyAsync(c->d_cnt_off.p, cnt_off.data(), sizeof(int64_t) * (nf + 1),
                          hipMemcpyHostToDevice, s));
    FT_HIP(hipStreamSynchronize(s));
    c->idx_G = G;
    for (int q = 0; q < kLevels; q++) c->idx_words[q] = q ? words[q] : G;
    c->idx_top = top;
    c->idx_layout = c->layout_gen;
    c->idx_bin_scale = bs;
    c->idx_reach = reach;
    return FT_OK;
}

inline int64_t at_least1(int64_t v) { return std::max<int64_t>(1, v); }

inline int64_t scan_blocks(int64_t n) { return std::max<int64_t>(1, (n + kScanTile - 1) / kScanTile); }

// Numbering of the index's leaves and nodes for at most n primitives: each
// level's capacity, and one more entry for the end of its last range.
struct LevelPlan {
    LevelOff lo;
    int64_t cap[kLevels];
    int64_t total;
};
LevelPlan level_plan(const ft_ctx* c, int64_t n)
{
    LevelPlan p{};
    int64_t at = 0;
    for (int k = 0; k < kLevels; k++) {
        p.cap[k] = std::min(n, c->idx_words[k]);
        p.lo.off[k] = (uint32_t)at;
        at += p.cap[k] + 1;
    }
    p.total = at;
    return p;
}

// The primitives' bins (later leaves) and places while the index is built: in
// the crossing tets' edges, which nothing reads once the triangles are made,
// where those are large enough (two entries a primitive; a tet has 16 bytes
// and at most two triangles).
struct PrimWork {
    uint32_t *code, *place;
};
bool prim_work_in_xedges(const ft_ctx* c, int64_t n) { return 2 * sizeof(uint32_t) * (size_t)n <= c->xedges.cap; }
PrimWork prim_work(const ft_ctx* c, int64_t n)
{
    if (!prim_work_in_xedges(c, n)) return {c->pcode.as<uint32_t>(), c->place.as<uint32_t>()};
    return {c->xedges.as<uint32_t>(), c->xedges.as<uint32_t>() + n};
}

// Device buffers of the stages of one reinit.  Stage 0: sized by the mesh;
// 1: by crossing tets and triangles; 2: by crossing points; 3: the index over
// n primitives (leaves <= min(bins, n)).
int ensure_stage(ft_ctx* c, int stage, const Caps& cp, int mode, bool want_nearest,
                 bool want_normals = false)
{
    const int64_t N = c->N, T = c->T, E = c->E, nf = c->nf;
    const int64_t nw_nodes = (N + 63) / 64, nw_tets = (T + 63) / 64, nw_edges = (E + 63) / 64;
    const int64_t nblk = (T + kBS - 1) / kBS;
    if (stage == 0) {
        FT_TRY(ensure(c->sbits, 8 * at_least1(nw_nodes)));
        FT_TRY(ensure(c->retain, 8 * at_least1(nw_nodes)));
        FT_TRY(ensure(c->tbits, 8 * at_least1(2 * nw_tets)));   // crossing, then two-triangle
        FT_TRY(ensure(c->blk, 8 * at_least1(nblk)));
        FT_TRY(ensure(c->ebits, 8 * at_least1(nw_edges)));
        FT_TRY(ensure(c->eprefix, 4 * at_least1(nw_edges)));
        FT_TRY(ensure(c->fcounts, sizeof(int64_t) * 3 * nf));
        FT_TRY(ensure(c->fclamp, sizeof(uint64_t) * nf));
        FT_TRY(ensure(c->roots, sizeof(uint32_t) * nf));
        if (want_nearest) FT_TRY(ensure(c->nearest, sizeof(int32_t) * at_least1(N)));
        if (want_normals) {
            FT_TRY(ensure(c->normals, 12 * at_least1(N)));
            FT_TRY(ensure(c->grad_t, 16 * at_least1(T)));
            FT_TRY(ensure(c->phi_ifn_int, 8 * at_least1(N)));
        }
    } else if (stage == 1) {
        FT_TRY(ensure(c->xtet, 4 * at_least1(cp.X)));
        FT_TRY(ensure(c->xtri_off, 4 * at_least1(cp.X)));
        FT_TRY(ensure(c->xedges, 16 * at_least1(cp.X)));
        FT_TRY(ensure(c->if_elems, 4 * at_least1(cp.X)));
        FT_TRY(ensure(c->tris, 16 * at_least1(cp.F)));
        FT_TRY(ensure(c->tri_norm, 4 * at_least1(cp.F)));
    } else if (stage == 2) {
        FT_TRY(ensure(c->ifp, 12 * at_least1(cp.P)));
        FT_TRY(ensure(c->ifp2e, 4 * at_least1(cp.P)));
        FT_TRY(ensure(c->ifp_area, 4 * at_least1(cp.P)));
        FT_TRY(ensure(c->p2t_off, 4 * (cp.P + 1)));
        FT_TRY(ensure(c->p2t_cursor, 4 * at_least1(cp.P)));
        FT_TRY(ensure(c->p2t, 4 * at_least1(3 * cp.F)));
        // the side stream's scans: the point lists, the tile schedule
        FT_TRY(ensure(c->scan_side, sizeof(uint64_t) * std::max(scan_blocks(cp.P), scan_blocks(c->n_slots / 64))));
    } else {
        const int64_t n = mode == 0 ? cp.P : cp.F;
        const int64_t W = c->idx_G / 64;
        const LevelPlan lp = level_plan(c, n);
        if (lp.total > (int64_t)UINT32_MAX)
            return ft::set_error(FT_ERR_ARG, "index: too many leaves (%lld)", (long long)lp.total);
        FT_TRY(ensure(c->bbits, 8 * at_least1(W)));
        FT_TRY(ensure(c->bprefix, 4 * at_least1(W)));
        if (!prim_work_in_xedges(c, n)) {
            FT_TRY(ensure(c->pcode, sizeof(uint32_t) * at_least1(n)));
            FT_TRY(ensure(c->place, sizeof(uint32_t) * at_least1(n)));
        }
        FT_TRY(ensure(c->pidx, sizeof(int32_t) * at_least1(n)));
        if (mode == 0) FT_TRY(ensure(c->prec, sizeof(float4) * at_least1(n)));
        else FT_TRY(ensure(c->trec, sizeof(TriRec) * at_least1(n)));
        FT_TRY(ensure(c->leaf_cnt, sizeof(uint32_t) * at_least1(lp.cap[0])));
        FT_TRY(ensure(c->leaf_bin, sizeof(uint32_t) * at_least1(lp.cap[0])));
        FT_TRY(ensure(c->nfirst, sizeof(uint32_t) * (lp.total + 64)));   // (read a wave at a time)
        FT_TRY(ensure(c->nitem, sizeof(Item) * (lp.total + 4)));
        FT_TRY(ensure(c->naxis, sizeof(float4) * lp.total));
        // scan scratch of the largest scan of a reinit
        const int64_t nb = std::max({scan_blocks(nblk), scan_blocks(nw_edges), scan_blocks(cp.P), scan_blocks(W),
                                     3 * scan_blocks(lp.cap[0])});
        FT_TRY(ensure(c->scan_bsum, sizeof(uint64_t) * nb));
        FT_TRY(ensure(c->deep_part, sizeof(ulonglong2) * 64 * kSplitParts * at_least1(split_tiles_cap(c->n_slots / 64))));
        // last, as the search does without them when the scratch has no room
        // (a dense interface in large bins: 56^3 with 0.74M triangles in bins of
        // two spacings takes 159 MiB with them, 114 without)
        const size_t titems = sizeof(Item) * (size_t)(n + 4);        // the search reads items by fours
        if (mode == 1 && !has_room(c->titem, titems)) c->titem = DevBuf{};
        else if (mode == 1) FT_TRY(ensure(c->titem, titems));
    }
    return FT_OK;
}

// The error word of the reinit (S_ERR) as a status.
int stage_error(uint64_t ev, ft_counts* cnt)
{
    if (ev == ~0ull) return FT_OK;
    cnt->bad_tet = (int64_t)(ev & ((1ull << 40) - 1));
    if ((ev >> 40) == (uint64_t)ftp::kErrIndex)
        return ft::set_error(FT_ERR_INTERNAL,
                             "interface index out of range at triangle or point %lld: the "
                             "point -> triangle stage stopped before writing",
                             (long long)cnt->bad_tet);
    if ((ev >> 40) == 1)
        return ft::set_error(FT_ERR_T2E,
                             "tet %lld: crossing edges from t2e do not match its node signs "
                             "(LevelSet.cpp:400-405)", (long long)cnt->bad_tet);
    return ft::set_error(FT_ERR_DEGENERATE,
                         "tet %lld crosses the interface but all its nodes have |phi| <= "
                         "FLT_MIN (LevelSet.cpp:338-341)", (long long)cnt->bad_tet);
}

// Node -> tets lists of the current fields (once per field layout; not in a
// captured graph: it synchronises).
int build_node_tets(ft_ctx* c, hipStream_t s)
{
    FT_TRY(materialize_conn(c));
    if (c->n2t_layout == c->layout_gen) return FT_OK;
    const int64_t N = c->N, T = c->T;
    FT_TRY(ensure(c->n2t_off, sizeof(uint64_t) * (N + 1)));
    FT_TRY(ensure(c->n2t_ids, sizeof(int32_t) * (4 * T + kNodeGather)));
    FT_TRY(ensure(c->pcode, sizeof(uint32_t) * at_least1(N)));          // counters
    uint32_t* cnt = c->pcode.as<uint32_t>();
    uint64_t* off = c->n2t_off.as<uint64_t>();
    // raised in the pinned mirror, read after the wait below
    unsigned long long* twice = reinterpret_cast<unsigned long long*>(c->h_scalars) + S_P2T;
    *twice = 0ull;
    FT_TRY(fill<uint32_t>(s, cnt, N, 0u));
    if (T > 0) hipLaunchKernelGGL(k_n2t_count, dim3(grid1d(T)), dim3(kBS), 0, s, c->tets.as<int4>(), T, cnt, twice);
    FT_TRY(scan<uint32_t, uint64_t>(c, s, cnt, off, N, off + N, LoadClear{}));   // cnt: then the fill's cursors
    if (T > 0)
        hipLaunchKernelGGL(k_n2t_fill, dim3(grid1d(T)), dim3(kBS), 0, s, c->tets.as<int4>(), T, off, cnt,
                           c->n2t_ids.as<int32_t>());
    if (N > 0) hipLaunchKernelGGL(k_n2t_sort, dim3(grid1d(N)), dim3(kBS), 0, s, off, N, c->n2t_ids.as<int32_t>());
    FT_TRY(check_launch());
    FT_HIP(hipStreamSynchronize(s));
    c->tets_twice = *(volatile unsigned long long*)twice != 0ull;
    c->n2t_layout = c->layout_gen;
    return FT_OK;
}

// What the search of a reinit reads and writes.
struct SearchSpec {
    int mode = 0;                    // 0: crossing points, 1: triangles
    float band = 0.0f;
    const double* phi_old = nullptr;
    double* phi_out = nullptr;
    double* phi_ifn = nullptr;
    bool use_retain = false;         // keep phi_old at crossing-edge nodes (update blend)
    int epi = EPI_RAW;
    double w_phi = 0.0, w_ifn = 0.0;
    bool want_nearest = false;
    bool want_normals = false;       // Assembler::grad_nodes of phi_ifn after the epilogue
    bool int_ifn = false;            // phi_ifn into the handle's buffer (normals need it)
    int query_block = 0;
    int waves_per_simd = 6;          // launch bound of the query (triangles: 5..8)
    bool whole_tiles = false;        // no tile is split over waves
};

// Copies of the resident meshes ms into the handle's concatenated arrays,
// one gather launch per array over all fields: the node coordinates and
// query slots (perm with padding kept at -1, sx, sy, sz as bit copies, the
// tile -> field map as constants), or with conn the tets, t2e and edges
// (offset to global ids).  Their piece tables go up in one copy.
int gather_meshes(ft_ctx* h, const std::vector<std::shared_ptr<ft_ctx>>& ms, hipStream_t s, bool conn)
{
    enum { G_XYZ, G_PERM, G_SX, G_SY, G_SZ, G_TILE, G_TET, G_T2E, G_EDGE, G_N };
    const int g0 = conn ? G_TET : G_XYZ, g1 = conn ? G_N : G_TET;
    const int nf = (int)ms.size();
    const size_t tab = (size_t)(3 * nf + 1);             // src pointers (nf), offsets (nf+1), adds (nf)
    std::vector<int64_t> host((size_t)(g1 - g0) * tab);
    for (int g = g0; g < g1; g++) {
        int64_t* t = host.data() + (g - g0) * tab;
        const int32_t** srcp = reinterpret_cast<const int32_t**>(t);
        int64_t* off = t + nf;
        int64_t* add = t + 2 * nf + 1;
        off[0] = 0;
        for (int k = 0; k < nf; k++) {
            const ft_ctx* m = ms[k].get();
            int64_t cnt = 0, a = 0;
            const void* src = nullptr;
            switch (g) {
            case G_XYZ: src = m->xyz.p; cnt = 3 * m->N; break;
            case G_PERM: src = m->perm.p; cnt = m->n_slots; a = h->node_off[k]; break;
            case G_SX: src = m->sx.p; cnt = m->n_slots; break;
            case G_SY: src = m->sy.p; cnt = m->n_slots; break;
            case G_SZ: src = m->sz.p; cnt = m->n_slots; break;
            case G_TILE: src = nullptr; cnt = m->n_slots / 64; a = k; break;
            case G_TET: src = m->tets.p; cnt = 4 * m->T; a = h->node_off[k]; break;
            case G_T2E: src = m->t2e.p; cnt = 6 * m->T; a = h->edge_off[k]; break;
            default: src = m->edges.p; cnt = 2 * m->E; a = h->node_off[k]; break;
            }
            srcp[k] = static_cast<const int32_t*>(src);
            off[k + 1] = off[k] + cnt;
            add[k] = a;
        }
    }
    FT_TRY(ensure(h->gather_tab, sizeof(int64_t) * host.size()));
    FT_HIP(hipMemcpyAsync(h->gather_tab.p, host.data(), sizeof(int64_t) * host.size(), hipMemcpyHostToDevice, s));
    void* dsts[G_N] = {h->xyz.p, h->perm.p, h->sx.p, h->sy.p, h->sz.p, h->tile_field.p, h->tets.p, h->t2e.p,
                       h->edges.p};
    for (int g = g0; g < g1; g++) {
        const int64_t* t = h->gather_tab.as<int64_t>() + (g - g0) * tab;
        const int64_t total = host[(g - g0) * tab + 2 * nf];
        if (total == 0) continue;
        hipLaunchKernelGGL(k_gather, dim3(grid1d(total, kGatherChunk)), dim3(kBS), 0, s,
                           reinterpret_cast<const int32_t* const*>(t), t + nf, t + 2 * nf + 1, nf,
                           g == G_PERM ? 1 : 0, static_cast<int32_t*>(dsts[g]));
    }
    FT_TRY(check_launch());
    // the host tables must outlive their (possibly staged) copy
    FT_HIP(hipStreamSynchronize(s));
    return FT_OK;
}

// The concatenated tets, t2e and edges of a batch of resident meshes, for the
// operations that index them globally (normals, curvature, surface tension,
// advection, ft_get_mesh); a no-op for any other handle.
int materialize_conn(ft_ctx* h)
{
    if (!h->virt) return FT_OK;
    drop_graph(h);                   // captured with the per-field view
    FT_TRY(ensure(h->tets, 16 * std::max<int64_t>(1, h->T)));
    FT_TRY(ensure(h->edges, 8 * std::max<int64_t>(1, h->E)));
    FT_TRY(ensure(h->t2e, 24 * std::max<int64_t>(1, h->T)));
    FT_TRY(gather_meshes(h, h->field_meshes, h->stream, true));
    h->virt = false;
    h->field_meshes.clear();
    return FT_OK;
}

MeshView mesh_view(ft_ctx* c)
{
    MeshView m{};
    m.nf = c->nf;
    m.node_off = c->d_node_off.as<int64_t>();
    m.tet_off = c->d_tet_off.as<int64_t>();
    m.edge_off = c->d_edge_off.as<int64_t>();
    if (!c->virt) {
        m.tets = c->tets.as<int4>();
        m.t2e3 = c->t2e.as<int2>();
        m.edges = c->edges.as<int2>();
    } else {
        const void* const* tab = static_cast<const void* const*>(c->field_tab.p);
        m.f_tets = reinterpret_cast<const int4* const*>(tab);
        m.f_t2e3 = reinterpret_cast<const int2* const*>(tab + c->nf);
        m.f_edges = reinterpret_cast<const int2* const*>(tab + 2 * c->nf);
    }
    return m;
}

// Enqueues the marching tets of one reinit on stream s.  eager: reads the
// stage totals back after the two counting scans (sizing the buffers exactly,
// and stopping early on a failed stage).  !eager (graph capture): no host
// reads and no allocation; the buffers were sized for `cp` beforehand and
// the kernels guard them (outgrown()).  counts_only: stops once the totals are known
// (phi is not written).
// Work enqueued on c->side from now on runs after everything enqueued on s
// so far.
int side_fork(ft_ctx* c, hipStream_t s)
{
    FT_HIP(hipEventRecord(c->side_fork_ev, s));
    FT_HIP(hipStreamWaitEvent(c->side, c->side_fork_ev, 0));
    c->side_open = true;
    return FT_OK;
}

// Work enqueued on s from now on runs after everything enqueued on c->side.
int side_join(ft_ctx* c, hipStream_t s)
{
    if (!c->side_open) return FT_OK;
    c->side_open = false;
    FT_HIP(hipEventRecord(c->side_join_ev, c->side));
    FT_HIP(hipStreamWaitEvent(s, c->side_join_ev, 0));
    return FT_OK;
}

// Joins the side stream into s when it leaves scope (early returns included).
struct SideJoin {
    ft_ctx* c;
    hipStream_t s;
    ~SideJoin() { (void)side_join(c, s); }
};

int enqueue_marching(ft_ctx* c, hipStream_t s, double* phi, int mode, bool want_nearest,
                     bool want_normals, Caps& cp, bool eager, bool counts_only, ft_counts* cnt,
                     bool timed)
{
    const int64_t N = c->N, T = c->T, E = c->E;
    uint64_t* sc = c->scalars.as<uint64_t>();
    const int64_t nw_tets = (T + 63) / 64, nw_edges = (E + 63) / 64;
    const int64_t nblk = (T + kBS - 1) / kBS;
    timed = timed && !counts_only;
    FT_TRY(ensure_stage(c, 0, cp, mode, want_nearest, want_normals));
    uint64_t* sbits = c->sbits.as<uint64_t>();
    if (timed) (void)hipEventRecord(c->ev[0], s);
    hipLaunchKernelGGL(k_node_signs, dim3(grid1d(N)), dim3(kBS), 0, s, phi, N, sbits,
                       c->retain.as<uint64_t>(), c->ebits.as<uint64_t>(), nw_edges, sc);
    if (T > 0)
        hipLaunchKernelGGL(k_classify, dim3((unsigned)((nblk + kClassifyGroups - 1) / kClassifyGroups)),
                           dim3(kBS), 0, s, mesh_view(c), T, sbits, c->tbits.as<uint64_t>(),
                           c->tbits.as<uint64_t>() + nw_tets, c->blk.as<uint64_t>());
    FT_TRY(scan<uint64_t, uint64_t>(c, s, c->blk.as<uint64_t>(), c->blk.as<uint64_t>(), nblk,
                                    sc + S_BLK, LoadSame{}));
    if (eager) {
        FT_TRY(read_scalars(c, s, S_TOP));
        cp.X = (int64_t)(c->h_scalars[S_BLK] >> 32);
        cp.F = (int64_t)(c->h_scalars[S_BLK] & 0xffffffffull);
        cnt->n_if_elems = cp.X;
        cnt->n_tri = cp.F;
    }
    FT_TRY(ensure_stage(c, 1, cp, mode, want_nearest));
    if (nw_tets > 0)
        hipLaunchKernelGGL(k_compact, dim3(grid1d(nw_tets)), dim3(kBS), 0, s, c->tbits.as<uint64_t>(),
                           c->tbits.as<uint64_t>() + nw_tets, nw_tets, c->blk.as<uint64_t>(),
                           c->xtet.as<int32_t>(), c->xtri_off.as<int32_t>(), sc, eager ? -1 : cp.X, eager ? -1 : cp.F);
    if (cp.X > 0)
        hipLaunchKernelGGL(k_xtet, dim3(grid1d(cp.X)), dim3(kBS), 0, s, c->tbits.as<uint64_t>() + nw_tets,
                           mesh_view(c), sbits, c->xtet.as<int32_t>(), sc,
                           c->ebits.as<unsigned long long>(), c->xedges.as<int4>());
    FT_TRY(scan<uint64_t, uint32_t>(c, s, c->ebits.as<uint64_t>(), c->eprefix.as<uint32_t>(),
                                    nw_edges, reinterpret_cast<uint32_t*>(sc + S_EDGES), LoadPopc{}));
    if (eager) {
        FT_TRY(read_scalars(c, s, S_TOP));
        cp.P = (int64_t)(c->h_scalars[S_EDGES] & 0xffffffffull);
        cnt->n_ifp = cp.P;
        FT_TRY(stage_error(c->h_scalars[S_ERR], cnt));
        if (counts_only) return FT_OK;
    }
    FT_TRY(ensure_stage(c, 2, cp, mode, want_nearest));
    if (nw_edges > 0)
        hipLaunchKernelGGL(k_points, dim3(grid1d(nw_edges)), dim3(kBS), 0, s, c->ebits.as<uint64_t>(),
                           c->eprefix.as<uint32_t>(), nw_edges, mesh_view(c), c->xyz.as<float>(),
                           phi, c->ifp.as<float>(), c->ifp2e.as<int32_t>(),
                           c->retain.as<unsigned long long>(), sc, eager ? -1 : cp.P);
    if (cp.X > 0)
        hipLaunchKernelGGL(k_tris, dim3(grid1d(cp.X)), dim3(kBS), 0, s, mesh_view(c), c->xyz.as<float>(),
                           phi, c->xtet.as<int32_t>(), c->xtri_off.as<int32_t>(), c->xedges.as<int4>(),
                           c->ebits.as<uint64_t>(), c->eprefix.as<uint32_t>(), c->ifp.as<float>(),
                           c->tris.as<int4>(), c->tri_norm.as<float>(), c->if_elems.as<int32_t>(), sc);
    // p2t and areas; entries past the point count stay empty.  The query
    // reads neither: they run on the side stream, beside the index build,
    // and the query's stream joins it before the query.
    FT_TRY(side_fork(c, s));
    {
        hipStream_t ss = c->side;
        uint32_t* deg = c->p2t_cursor.as<uint32_t>();
        FT_TRY(fill<uint32_t>(ss, deg, cp.P, 0u));
        if (cp.F > 0)
            hipLaunchKernelGGL(k_p2t_count, dim3(grid1d(cp.F)), dim3(kBS), 0, ss, c->tris.as<int4>(), sc, deg);
        // deg: the degrees, then (cleared by the scan) the fill's cursors
        FT_TRY(scan<uint32_t, uint32_t>(c, ss, deg, c->p2t_off.as<uint32_t>(), cp.P,
                                        c->p2t_off.as<uint32_t>() + cp.P, LoadClear{}, &c->scan_side));
        if (cp.F > 0)
            hipLaunchKernelGGL(k_p2t_fill, dim3(grid1d(cp.F)), dim3(kBS), 0, ss, c->tris.as<int4>(), sc,
                               c->p2t_off.as<uint32_t>(), deg, c->p2t.as<int32_t>());
        if (cp.P > 0)
            hipLaunchKernelGGL(k_point_area, dim3(grid1d(cp.P)), dim3(kBS), 0, ss, c->p2t_off.as<uint32_t>(),
                               sc, c->p2t.as<int32_t>(), c->tri_norm.as<float>(), c->ifp_area.as<float>());
    }
    if (c->nf > 1)
        hipLaunchKernelGGL(k_field_counts, dim3((c->nf + 63) / 64), dim3(64), 0, s, c->nf,
                           c->d_tet_off.as<int64_t>(), c->d_edge_off.as<int64_t>(), T, E,
                           c->tbits.as<uint64_t>(), c->blk.as<uint64_t>(), c->xtri_off.as<int32_t>(),
                           c->ebits.as<uint64_t>(), c->eprefix.as<uint32_t>(), sc,
                           c->fcounts.as<int64_t>());
    FT_TRY(check_launch());
    if (timed) (void)hipEventRecord(c->ev[1], s);
    // a degenerate tet found by k_tris halts the rest on the device; the final
    // readback reports it
    return FT_OK;
}

// The query kernel for (mode, threads per workgroup, waves per SIMD); points
// mode has its best bound only.  Eight runs as seven, which is what the waves'
// LDS admits: bounded at eight the compiler gives the bound up and takes 94
// registers, four waves (96^3 triangles 0.835 ms; 0.758 at seven, 0.736 at six).
template <int MODE, int BS>
int launch_query_bs(int wps, dim3 g, dim3 b, hipStream_t s, const QueryArgs& q)
{
    switch (MODE == 0 ? 6 : wps) {
    case 5: hipLaunchKernelGGL((k_query_wave<MODE, BS, MODE == 0 ? 6 : 5>), g, b, 0, s, q); break;
    case 7: hipLaunchKernelGGL((k_query_wave<MODE, BS, MODE == 0 ? 6 : 7>), g, b, 0, s, q); break;
    default: hipLaunchKernelGGL((k_query_wave<MODE, BS, 6>), g, b, 0, s, q); break;
    }
    return check_launch();
}

int launch_query(int mode, int qb, int wps, dim3 g, dim3 b, hipStream_t s, const QueryArgs& q)
{
    if (mode == 1 && !q.titem) {                      // (qb is 64)
        hipLaunchKernelGGL((k_query_wave<1, 64, 6, false, true>), g, b, 0, s, q);
        return check_launch();
    }
    if (q.stats) {                                    // counting build (qb is 64)
        if (mode == 0) hipLaunchKernelGGL((k_query_wave<0, 64, 5, true>), g, b, 0, s, q);
        else hipLaunchKernelGGL((k_query_wave<1, 64, 5, true>), g, b, 0, s, q);
        return check_launch();
    }
    if (mode == 0) {
        if (qb == 64) return launch_query_bs<0, 64>(wps, g, b, s, q);
        if (qb == 128) return launch_query_bs<0, 128>(wps, g, b, s, q);
        return launch_query_bs<0, 256>(wps, g, b, s, q);
    }
    if (qb == 64) return launch_query_bs<1, 64>(wps, g, b, s, q);
    if (qb == 128) return launch_query_bs<1, 128>(wps, g, b, s, q);
    return launch_query_bs<1, 256>(wps, g, b, s, q);
}

// Enqueues the bin index over the primitives (crossing points c->ifp, or
// triangles c->tris) and the distance query with its epilogue.  The number of
// primitives is read on the device (S_EDGES or S_BLK); cp bounds it.
int enqueue_search(ft_ctx* c, hipStream_t s, const SearchSpec& sp, const Caps& cp, bool eager,
                   bool timed)
{
    const int mode = sp.mode;
    uint64_t* sc = c->scalars.as<uint64_t>();
    (void)eager;
    const int64_t n_cap = mode == 0 ? cp.P : cp.F;
    const float* ifp = c->ifp.as<float>();
    const int4* tris = mode == 0 ? nullptr : c->tris.as<int4>();
    const int nf = c->nf;
    if (c->idx_layout != c->layout_gen)
        return ft::set_error(FT_ERR_STATE, "index grids not set up for this field layout");
    FT_TRY(ensure_stage(c, 3, cp, mode, sp.want_nearest));
    // Deep tiles first, in a full-domain search.  That schedule reads only phi
    // and the slots: it is built on the side stream while the index is built
    // here.  (A narrow band's follows the index, below.)
    const int64_t n_tiles = c->n_slots / 64;
    int32_t* tile_list = nullptr;
    // tile_sched: classes (u32), the launch order (i32), the scan (u64)
    uint32_t* cls = c->tile_sched.as<uint32_t>();
    uint64_t* ex = reinterpret_cast<uint64_t*>(cls + 2 * n_tiles);
    if (n_tiles > 0) tile_list = reinterpret_cast<int32_t*>(cls + n_tiles);
    if (sp.band <= 0.0f && n_tiles > 0) {
        FT_TRY(side_fork(c, s));
        hipStream_t ss = c->side;
        hipLaunchKernelGGL(k_tile_deep, dim3(grid1d(64 * n_tiles)), dim3(kBS), 0, ss, n_tiles,
                           c->perm.as<int32_t>(), sp.phi_old, c->tile_field.as<int32_t>(),
                           c->d_grids.as<Grid>(), kDeepTile * split_tile_h(n_tiles), split_tile_h(n_tiles), cls, sc);
        FT_TRY(scan<uint32_t, uint64_t>(c, ss, cls, ex, n_tiles, sc + S_DEEP, LoadTileClass{}, &c->scan_side));
        hipLaunchKernelGGL(k_tile_list, dim3(grid1d(n_tiles)), dim3(kBS), 0, ss, n_tiles, cls, ex, sc,
                           tile_list);
    }
    const int64_t W = c->idx_G / 64;
    const LevelPlan lp = level_plan(c, n_cap);
    const IndexGeom ig{c->d_edge_off.as<int64_t>(), c->d_cnt_off.as<int64_t>(), c->d_grids.as<Grid>(), nf};
    uint64_t* bits = c->bbits.as<uint64_t>();
    uint32_t* lcnt = c->leaf_cnt.as<uint32_t>();
    uint32_t* lbin = c->leaf_bin.as<uint32_t>();
    uint32_t* first = c->nfirst.as<uint32_t>();
    const PrimWork work = prim_work(c, n_cap);
    uint64_t* clamped = nf == 1 ? sc + S_CLAMP : c->fclamp.as<uint64_t>();
    WordRanges clr;
    clr.add(bits, 2 * W, 0u);
    clr.add(lcnt, lp.cap[0], 0u);
    clr.add(c->roots.p, nf, ~0u);
    clr.add(sc + S_BINS, 2, 0u);                       // the bitmap scan writes the low 32 bits
    clr.add(clamped, 2 * nf, 0u);
    clr.add(sc + S_Q, 9 * kQueueLine, 0u);
    if (sp.band > 0.0f) clr.add(sc + S_DEEP, 2, 0u);
    FT_TRY(set_words(s, clr));
    if (n_cap > 0) {
        hipLaunchKernelGGL(k_prim_bin, dim3(grid1d(n_cap)), dim3(kBS), 0, s, mode, sc, ifp, tris,
                           nf > 1 ? c->ifp2e.as<int32_t>() : nullptr, ig, work.code, (unsigned long long*)bits);
        FT_TRY(scan<uint64_t, uint32_t>(c, s, bits, c->bprefix.as<uint32_t>(), W,
                                        reinterpret_cast<uint32_t*>(sc + S_BINS), LoadPopc{}));
        hipLaunchKernelGGL(k_prim_rank, dim3(grid1d(n_cap)), dim3(kBS), 0, s, mode, sc, bits,
                           c->bprefix.as<uint32_t>(), work.code, work.place, lcnt, lbin);
        if (lp.cap[0] <= kLevelOne) {
            hipLaunchKernelGGL(k_level_one, dim3(1), dim3(1024), 0, s, sc, lcnt, lbin, ig, lp.lo, first,
                               c->roots.as<uint32_t>());
        } else {
            const int64_t nb = scan_blocks(lp.cap[0]);
            ftd::Lv* bs = c->scan_bsum.as<ftd::Lv>();
            hipLaunchKernelGGL(k_level_reduce, dim3((unsigned)nb), dim3(kBS), 0, s, sc, lcnt, lbin, ig, bs);
            hipLaunchKernelGGL(k_scan_top<ftd::Lv>, dim3(1), dim3(1024), 0, s, bs, nb,
                               reinterpret_cast<ftd::Lv*>(sc + S_LV));
            hipLaunchKernelGGL(k_level_down, dim3((unsigned)nb), dim3(kBS), 0, s, sc, lcnt, lbin, ig, bs, lp.lo, first,
                               c->roots.as<uint32_t>());
        }
        hipLaunchKernelGGL(k_prim_scatter, dim3(grid1d(n_cap)), dim3(kBS), 0, s, mode, sc, ifp, tris, work.code,
                           work.place, first, lbin, ig, c->prec.as<float4>(), c->titem.as<Item>(),
                           c->trec.as<TriRec>(), c->pidx.as<int32_t>());
        hipLaunchKernelGGL(mode == 0 ? k_leaf_items<0> : k_leaf_items<1>, dim3(grid1d(kLeafLanes * lp.cap[0])),
                           dim3(kBS), 0, s, sc, first, lbin, ig, c->pidx.as<int32_t>(), ifp, tris,
                           c->nitem.as<Item>(), c->naxis.as<float4>());
        for (int k = 1; k < c->idx_top; k++)               // a root's own box is never tested
            hipLaunchKernelGGL(k_node_items, dim3((unsigned)std::min<int64_t>(grid1d(64 * lp.cap[k]), kNodeBlocks)),
                               dim3(kBS), 0, s, sc, k, lp.lo.off[k], first, c->nitem.as<Item>(), c->naxis.as<float4>());
    }
    FT_TRY(check_launch());

    // ---- distance query with the fused epilogue --------------------------------
    QueryArgs q{};
    q.n_slots = c->n_slots;
    q.sx = c->sx.as<float>(); q.sy = c->sy.as<float>(); q.sz = c->sz.as<float>();
    q.perm = c->perm.as<int32_t>();
    q.tile_field = c->tile_field.as<int32_t>();
    q.grids = c->d_grids.as<Grid>();
    q.roots = c->roots.as<uint32_t>();
    q.first = first;
    q.items = c->nitem.as<Item>();
    q.leaf_end = lp.lo.off[1];
    q.prec = c->prec.as<float4>();
    q.titem = c->titem.as<Item>();
    q.trec = c->trec.as<TriRec>();
    q.band = sp.band;
    q.ifp = ifp;
    q.tris = tris;
    q.phi_old = sp.phi_old;
    q.phi_out = sp.phi_out;
    q.phi_ifn = sp.phi_ifn ? sp.phi_ifn : (sp.int_ifn ? c->phi_ifn_int.as<double>() : nullptr);
    q.retain = sp.use_retain ? c->retain.as<uint64_t>() : nullptr;   // resolved after allocation
    q.nearest = sp.want_nearest ? c->nearest.as<int32_t>() : nullptr;
    q.epi = sp.epi;
    q.w_phi = sp.w_phi;
    q.w_ifn = sp.w_ifn;
    // (the schedule's scan, which nothing reads any more)
    q.clamped = reinterpret_cast<uint32_t*>(ex);
    static const bool want_stats = getenv("FT_QUERY_STATS") != nullptr;
    q.h_est = c->h_est;
    if (want_stats && eager) {
        FT_TRY(ensure(c->stats, 8 * 48));
        FT_TRY(fill<uint64_t>(s, c->stats.as<uint64_t>(), 48, 0ull));
        q.stats = c->stats.as<unsigned long long>();
    }
    // the first search for each tile's centre; in a narrow band too (128^3
    // star, 6 h: surface tiles test half the leaves and a third of the pairs,
    // query 0.597 -> 0.511 ms)
    q.probe = !(getenv("FT_PROBE") && !strcmp(getenv("FT_PROBE"), "0"));
    q.sc = sc;
    if (timed) (void)hipEventRecord(c->ev[2], s);
    FT_TRY(side_join(c, s));                          // the schedule and the point lists
    if (tile_list) {
        q.tile_list = tile_list;
        q.n_deep = sc + S_DEEP;
    }
    if (c->n_slots > 0 && sp.band > 0.0f) {
        hipLaunchKernelGGL(k_tile_near, dim3(grid1d(n_tiles, 64)), dim3(64), 0, s, q, lp.lo.off[2], cls, tile_list,
                           (unsigned long long*)(sc + S_DEEP));
        // the others beside the search of those
        FT_TRY(side_fork(c, s));
        hipLaunchKernelGGL(mode == 0 ? k_far_tiles<0> : k_far_tiles<1>, dim3(grid1d(64 * n_tiles)), dim3(kBS), 0,
                           c->side, q, cls);
        FT_TRY(check_launch());
    }
    if (c->n_slots > 0) {
        const bool records = mode == 1 && !q.titem;
        const int qb = q.stats || records || sp.query_block == 0 ? 64 : sp.query_block;
        const int wps = mode == 0 || records ? 6 : std::min(sp.waves_per_simd, 7);
        if (sp.band <= 0.0f && !sp.whole_tiles) q.split_out = c->deep_part.as<ulonglong2>();
        // as many waves as the device holds at this launch bound (4 SIMDs per
        // CU), or as there may be tiles and parts; whole workgroups
        const int64_t items = n_tiles + (q.split_out ? split_tiles_cap(n_tiles) * (kSplitParts - 1) : 0);
        const int64_t waves = std::min<int64_t>((int64_t)c->cu_count * 4 * wps, items);
        const dim3 g(grid1d(waves, qb / 64)), b(qb);
        q.queue = reinterpret_cast<uint32_t*>(sc + S_Q);
        FT_TRY(launch_query(mode, qb, wps, g, b, s, q));
        if (sp.band > 0.0f) {
            FT_TRY(side_join(c, s));
            hipLaunchKernelGGL(k_clamp_sum, dim3(grid1d((n_tiles + kClampRun - 1) / kClampRun * 64)), dim3(kBS), 0, s,
                               n_tiles, q.clamped, q.tile_field, reinterpret_cast<unsigned long long*>(clamped), sc);
            FT_TRY(check_launch());
        }
        if (q.split_out) {
            const dim3 gm(grid1d(64 * split_tiles_cap(n_tiles)));
            if (mode == 0) hipLaunchKernelGGL(k_split_merge<0>, gm, dim3(kBS), 0, s, q);
            else hipLaunchKernelGGL(k_split_merge<1>, gm, dim3(kBS), 0, s, q);
            FT_TRY(check_launch());
        }
    }
    if (timed) (void)hipEventRecord(c->ev[3], s);
    if (sp.want_normals && c->N > 0) {
        if (c->n2t_layout != c->layout_gen)
            return ft::set_error(FT_ERR_STATE, "node -> tets lists not built for this field layout");
        if (c->T > 0)
            hipLaunchKernelGGL(k_tet_grad, dim3(grid1d(c->T)), dim3(kBS), 0, s, c->tets.as<int4>(), c->T,
                               c->xyz.as<float>(), q.phi_ifn, c->grad_t.as<float4>(), sc);
        hipLaunchKernelGGL(k_node_normals, dim3(grid1d(c->N)), dim3(kBS), 0, s, c->n2t_off.as<uint64_t>(),
                           c->n2t_ids.as<int32_t>(), c->grad_t.as<float4>(), c->N, c->normals.as<float>(), sc);
        FT_TRY(check_launch());
    }
    if (timed) (void)hipEventRecord(c->ev[4], s);
    return FT_OK;
}

// After the reinit's kernels: totals, errors and per-field counts from the
// device (one readback).  Returns FT_ERR_BUDGET internally when a stage
// outgrew the capacities of a captured graph.
int collect(ft_ctx* c, hipStream_t s, bool want_nearest, ft_counts* cnt)
{
    const int nf = c->nf;
    FT_HIP(hipMemcpyAsync(c->h_scalars, c->scalars.p, sizeof(uint64_t) * S_TOP, hipMemcpyDeviceToHost, s));
    std::vector<uint64_t> clamp(nf);
    std::vector<int64_t> fc(nf > 1 ? 3 * nf : 0);
    if (nf > 1) {
        FT_HIP(hipMemcpyAsync(clamp.data(), c->fclamp.p, 8 * nf, hipMemcpyDeviceToHost, s));
        FT_HIP(hipMemcpyAsync(fc.data(), c->fcounts.p, sizeof(int64_t) * 3 * nf, hipMemcpyDeviceToHost, s));
    }
    FT_HIP(hipStreamSynchronize(s));
    const uint64_t* hs = c->h_scalars;
    if (nf == 1) clamp[0] = hs[S_CLAMP];
    *cnt = ft_counts{};
    cnt->n_if_elems = (int64_t)(hs[S_BLK] >> 32);
    cnt->n_tri = (int64_t)(hs[S_BLK] & 0xffffffffull);
    cnt->n_ifp = (int64_t)(hs[S_EDGES] & 0xffffffffull);
    cnt->bad_tet = -1;
    if (hs[S_CAP]) return FT_ERR_BUDGET;
    FT_TRY(stage_error(hs[S_ERR], cnt));
    c->have_interface = true;
    c->field_counts.assign(nf, ft_counts{});
    for (int k = 0; k < nf; k++) {
        ft_counts& f = c->field_counts[k];
        if (nf > 1) {
            f.n_ifp = fc[3 * k];
            f.n_tri = fc[3 * k + 1];
            f.n_if_elems = fc[3 * k + 2];
        } else {
            f = *cnt;
        }
        f.bad_tet = -1;
        f.n_clamped = (int64_t)clamp[k];
        cnt->n_clamped += f.n_clamped;
    }
    c->have_nearest = want_nearest;
    return FT_OK;
}

void print_query_stats(ft_ctx* c, int mode)
{
    uint64_t st[48];
    if (hipMemcpy(st, c->stats.p, sizeof st, hipMemcpyDeviceToHost) != hipSuccess) return;
    static const char* names[8] = {"out <2h", "out 2-8h", "out 8-32h", "out >32h",
                                   "in <2h", "in 2-8h", "in 8-32h", "in >32h"};
    static const char* what = "nodes %.1f boxes %.1f leaves %.1f primitives %.1f pairs %.1f\n";
    double t[6] = {0, 0, 0, 0, 0, 0};
    for (int b = 0; b < 8; b++)
        for (int q = 0; q < 6; q++) t[q] += (double)st[6 * b + q];
    // the counts are the tile's, added once per node
    fprintf(stderr, "[ftreinit] query mode %d: N=%lld, per tile: ", mode, (long long)c->N);
    fprintf(stderr, what, t[1] / t[0], t[2] / t[0], t[3] / t[0], t[4] / t[0], t[5] / t[0]);
    for (int b = 0; b < 8; b++) {
        const double nn = (double)st[6 * b];
        if (!(nn > 0)) continue;
        fprintf(stderr, "[ftreinit]   %-9s %5.1f%% of nodes: ", names[b], 100.0 * nn / c->N);
        fprintf(stderr, what, st[6 * b + 1] / nn, st[6 * b + 2] / nn, st[6 * b + 3] / nn, st[6 * b + 4] / nn,
                st[6 * b + 5] / nn);
    }
}

SearchSpec reinit_search_spec(double* phi, double* phi_ifn, const ft_opts* o)
{
    SearchSpec sp;
    sp.mode = o->mode == FT_DIST_POINTS ? 0 : 1;
    sp.band = (float)o->band;
    sp.phi_old = phi;
    sp.phi_out = phi;                // read and written per node in place
    sp.phi_ifn = phi_ifn;
    sp.use_retain = true;
    sp.epi = (o->blend == FT_BLEND_INIT) ? EPI_INIT : EPI_UPDATE;
    sp.w_phi = o->w_phi;
    sp.w_ifn = o->w_ifn;
    sp.want_nearest = o->want_nearest != 0;
    sp.want_normals = o->want_normals != 0;
    sp.int_ifn = sp.want_normals && !phi_ifn;
    sp.query_block = o->query_block;
    sp.waves_per_simd = o->waves_per_simd > 0 ? o->waves_per_simd : 6;
    sp.whole_tiles = o->schedule == FT_SCHED_QUEUE;
    return sp;
}

int validate_opts(const ft_opts* o)
{
    if (!o) return ft::set_error(FT_ERR_ARG, "null options");
    if (o->mode != FT_DIST_POINTS && o->mode != FT_DIST_TRIANGLES)
        return ft::set_error(FT_ERR_ARG, "unknown distance mode %d", o->mode);
    if (o->blend != FT_BLEND_INIT && o->blend != FT_BLEND_UPDATE)
        return ft::set_error(FT_ERR_ARG, "unknown blend %d", o->blend);
    if (!(o->band >= 0.0) || o->band > 1e30)
        return ft::set_error(FT_ERR_ARG, "band must be >= 0");
    if (!(o->bin_scale >= 0.0f) || o->bin_scale > 1e6f)
        return ft::set_error(FT_ERR_ARG, "bin_scale must be >= 0");
    if (o->query_block != 0 && o->query_block != 64 && o->query_block != 128 && o->query_block != 256)
        return ft::set_error(FT_ERR_ARG, "query_block must be 0, 64, 128 or 256");
    if (o->waves_per_simd != 0 && (o->waves_per_simd < 5 || o->waves_per_simd > 8))
        return ft::set_error(FT_ERR_ARG, "waves_per_simd must be 0 or 5..8");
    if (o->schedule != FT_SCHED_STATIC && o->schedule != FT_SCHED_QUEUE && o->schedule != FT_SCHED_BINS)
        return ft::set_error(FT_ERR_ARG, "unknown query schedule %d", o->schedule);
    if (o->schedule == FT_SCHED_BINS && !(o->band > 0.0 && o->mode == FT_DIST_TRIANGLES))
        return ft::set_error(FT_ERR_ARG, "the bins schedule is for a narrow band in triangles mode");
    return FT_OK;
}

// Capacity with headroom over a measured stage total.
inline int64_t with_room(int64_t v) { return v + v / 4 + 256; }

int reinit_device(ft_ctx* c, double* d_phi, double* d_phi_ifn, const ft_opts* o,
                  ft_counts* counts, hipStream_t s, bool allow_spec = true)
{
    FT_TRY(validate_opts(o));
    if (!c->has_conn) return ft::set_error(FT_ERR_STATE, "reinit before a mesh was set");
    if (!d_phi) return ft::set_error(FT_ERR_ARG, "null phi");
    c->have_interface = false;
    c->have_nearest = false;
    c->have_normals = false;
    ft_counts cnt{};
    cnt.bad_tet = -1;
    Caps cp;
    const SearchSpec sp = reinit_search_spec(d_phi, d_phi_ifn, o);
    SideJoin join{c, s};
    int rc = index_setup(c, s, o->bin_scale, sp.mode);
    if (rc == FT_OK && sp.want_normals) rc = build_node_tets(c, s);
    // Speculative pass: the capacities of the last call on these fields, no
    // readback between stages (the device guards them, and halts before phi is
    // written if a stage outgrows them); else, or then, the exact pass, which
    // reads the stage totals back to size the buffers.
    const bool spec = allow_spec && rc == FT_OK && c->spec_layout == c->layout_gen && c->spec_mode == sp.mode;
    if (spec) {
        cp = c->spec_caps;
        rc = enqueue_marching(c, s, d_phi, sp.mode, sp.want_nearest, sp.want_normals, cp, false, false,
                              &cnt, c->timing);
        if (rc == FT_OK) rc = enqueue_search(c, s, sp, cp, false, c->timing);
        if (rc == FT_OK) rc = collect(c, s, sp.want_nearest, &cnt);
        c->spec_hits += rc != FT_ERR_BUDGET;
    }
    if (!spec || rc == FT_ERR_BUDGET) {
        cp = Caps{};
        cnt = ft_counts{};
        cnt.bad_tet = -1;
        rc = index_setup(c, s, o->bin_scale, sp.mode);
        if (rc == FT_OK)
            rc = enqueue_marching(c, s, d_phi, sp.mode, sp.want_nearest, sp.want_normals, cp, true, false,
                                  &cnt, c->timing);
        if (rc == FT_OK) rc = enqueue_search(c, s, sp, cp, true, c->timing);
        if (rc == FT_OK) rc = collect(c, s, sp.want_nearest, &cnt);
        if (rc == FT_OK) {
            c->spec_caps.X = with_room(cp.X);
            c->spec_caps.F = with_room(cp.F);
            c->spec_caps.P = with_room(cp.P);
            c->spec_layout = c->layout_gen;
            c->spec_mode = sp.mode;
        }
    }
    c->have_normals = rc == FT_OK && sp.want_normals;
    c->last_phi = d_phi;
    if (counts) *counts = cnt;
    c->last = cnt;
    static const bool want_stats = getenv("FT_QUERY_STATS") != nullptr;
    if (rc == FT_OK && want_stats && c->N > 0) print_query_stats(c, sp.mode);
    if (rc == FT_OK && c->timing) {
        float ms[4] = {0, 0, 0, 0};
        (void)hipEventSynchronize(c->ev[4]);
        for (int k = 0; k < 4; k++) (void)hipEventElapsedTime(&ms[k], c->ev[k], c->ev[k + 1]);
        for (int k = 0; k < 4; k++) c->phase_ms[k] += ms[k];
        c->timed_calls++;
    }
    return rc;
}

// ----------------------------------------------------------------------------
// Graph form: the whole reinit of the resident fields as one captured graph
// ----------------------------------------------------------------------------
bool same_opts(const ft_opts& a, const ft_opts& b)
{
    return a.mode == b.mode && a.blend == b.blend && a.w_phi == b.w_phi && a.w_ifn == b.w_ifn &&
           a.band == b.band && a.bin_scale == b.bin_scale && a.want_nearest == b.want_nearest &&
           a.query_block == b.query_block && a.want_normals == b.want_normals &&
           a.waves_per_simd == b.waves_per_simd && a.schedule == b.schedule;
}

void drop_graph(ft_ctx* c)
{
    if (c->graph.exec) (void)hipGraphExecDestroy(c->graph.exec);
    if (c->graph.graph) (void)hipGraphDestroy(c->graph.graph);
    c->graph.exec = nullptr;
    c->graph.graph = nullptr;
}

// Captures the reinit of (d_phi, d_phi_ifn, o) with capacities cp on the
// handle's stream.  Everything it touches is allocated before the capture.
int capture_reinit(ft_ctx* c, double* d_phi, double* d_phi_ifn, const ft_opts* o, const Caps& cp)
{
    drop_graph(c);
    const SearchSpec sp = reinit_search_spec(d_phi, d_phi_ifn, o);
    if (sp.want_normals) FT_TRY(build_node_tets(c, c->stream));
    for (int st = 0; st < 4; st++) FT_TRY(ensure_stage(c, st, cp, sp.mode, sp.want_nearest, sp.want_normals));
    FT_HIP(hipStreamSynchronize(c->stream));
    FT_HIP(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    Caps cc = cp;
    ft_counts unused{};
    int rc = enqueue_marching(c, c->stream, d_phi, sp.mode, sp.want_nearest, sp.want_normals, cc, false,
                              false, &unused, false);
    if (rc == FT_OK) rc = enqueue_search(c, c->stream, sp, cc, false, false);
    const int rj = side_join(c, c->stream);          // the capture must end joined
    if (rc == FT_OK) rc = rj;
    hipGraph_t graph = nullptr;
    const hipError_t e = hipStreamEndCapture(c->stream, &graph);
    if (rc != FT_OK) {
        if (graph) (void)hipGraphDestroy(graph);
        return rc;
    }
    if (e != hipSuccess)
        return ft::set_error(FT_ERR_HIP, "hipStreamEndCapture failed: %s", hipGetErrorString(e));
    hipGraphExec_t exec = nullptr;
    const hipError_t ei = hipGraphInstantiateWithFlags(&exec, graph, 0);
    if (ei != hipSuccess) {
        (void)hipGraphDestroy(graph);
        return ft::set_error(FT_ERR_HIP, "hipGraphInstantiate failed: %s", hipGetErrorString(ei));
    }
    GraphState& g = c->graph;
    g.graph = graph;
    g.exec = exec;
    g.phi = d_phi;
    g.phi_ifn = d_phi_ifn;
    g.opts = *o;
    g.layout = c->layout_gen;
    g.caps = cp;
    g.bufs = buffer_addresses(c);
    g.captures++;
    return FT_OK;
}

// Reinit of the resident fields through a captured graph: the first call (or
// a call whose pointers, options, fields or buffer sizes differ from the
// captured ones) sizes the stages with a counting pass over phi, captures
// with headroom and launches; later calls launch the same graph.  A call
// whose interface outgrows the headroom is detected on the device (nothing
// is written), captured again with room for it, and launched again.
int reinit_graph(ft_ctx* c, double* d_phi, double* d_phi_ifn, const ft_opts* o, ft_counts* counts,
                 hipStream_t s)
{
    FT_TRY(validate_opts(o));
    if (!c->has_conn) return ft::set_error(FT_ERR_STATE, "reinit before a mesh was set");
    if (!d_phi) return ft::set_error(FT_ERR_ARG, "null phi");
    c->have_interface = false;
    c->have_nearest = false;
    c->have_normals = false;
    GraphState& g = c->graph;
    ft_counts cnt{};
    cnt.bad_tet = -1;
    FT_TRY(index_setup(c, s, o->bin_scale, o->mode == FT_DIST_POINTS ? 0 : 1));
    const bool same = g.exec && g.phi == d_phi && g.phi_ifn == d_phi_ifn && same_opts(g.opts, *o) &&
                      g.layout == c->layout_gen;
    Caps cp = g.caps;
    bool fresh = !same;
    if (fresh) {
        Caps exact;
        const int mode = o->mode == FT_DIST_POINTS ? 0 : 1;
        const int rc = enqueue_marching(c, s, d_phi, mode, o->want_nearest != 0, o->want_normals != 0,
                                        exact, true, true, &cnt, false);
        if (rc != FT_OK) {
            if (counts) *counts = cnt;
            c->last = cnt;
            return rc;
        }
        cp.X = with_room(exact.X);
        cp.F = with_room(exact.F);
        cp.P = with_room(exact.P);
    }
    for (int attempt = 0; attempt < 4; attempt++) {
        if (fresh || buffer_addresses(c) != g.bufs) FT_TRY(capture_reinit(c, d_phi, d_phi_ifn, o, cp));
        FT_HIP(hipGraphLaunch(g.exec, s));
        g.launches++;
        const int rc = collect(c, s, o->want_nearest != 0, &cnt);
        c->have_normals = rc == FT_OK && o->want_normals != 0;
        c->last_phi = d_phi;
        if (rc != FT_ERR_BUDGET) {
            if (counts) *counts = cnt;
            c->last = cnt;
            return rc;
        }
        // Outgrown: the totals of the stages that ran are this call's.
        const uint64_t why = c->h_scalars[S_CAP];
        cp.X = std::max(cp.X, with_room(cnt.n_if_elems));
        cp.F = std::max(cp.F, with_room(cnt.n_tri));
        if (why & 2ull) cp.P = std::max(cp.P, with_room(cnt.n_ifp));
        fresh = true;
    }
    return ft::set_error(FT_ERR_HIP, "graph reinit: stage capacities did not settle");
}

std::mutex g_create_mu;

// ---- allocation-free reinit ---------------------------------------------------
// Per-call workspaces of ft_reinit_device_noalloc: one file-scope device array
// per GPU, held by every process that loads the library until it ends.  Its
// device address comes from hipGetSymbolAddress, once per device (the host
// name `scratch` is only a stand-in, not an address a kernel may use).
constexpr size_t kScratchBytes = size_t(FT_NOALLOC_SCRATCH_BYTES);
static __device__ __align__(256) unsigned char scratch[kScratchBytes];
std::mutex g_scratch_mu;
std::vector<void*> g_scratch_ptr;    // per device; null until looked up

int scratch_address(int device, void** out)
{
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if ((int)g_scratch_ptr.size() <= device) g_scratch_ptr.resize(device + 1, nullptr);
    if (!g_scratch_ptr[device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));   // device is current
        if (e != hipSuccess || !p)
            return ft::set_error(FT_ERR_HIP, "hipGetSymbolAddress(scratch) failed: %s",
                                 hipGetErrorString(e));
        g_scratch_ptr[device] = p;
    }
    *out = g_scratch_ptr[device];
    return FT_OK;
}

// The handle's per-call buffers (everything but the resident mesh, its query
// slots and tile lists, and the small scalars).
std::vector<DevBuf*> call_buffers(ft_ctx* h)
{
    return {&h->phi_tmp, &h->phi_ifn_tmp, &h->sbits, &h->retain, &h->tbits, &h->blk, &h->xtet,
            &h->xtri_off, &h->xedges, &h->ebits, &h->eprefix, &h->ifp, &h->ifp2e, &h->tris,
            &h->tri_norm, &h->if_elems, &h->p2t_off, &h->p2t_cursor, &h->p2t, &h->ifp_area,
            &h->nearest, &h->fcounts, &h->fclamp, &h->normals, &h->grad_t, &h->phi_ifn_int,
            &h->bbits, &h->bprefix, &h->pcode, &h->place, &h->prec, &h->titem, &h->trec, &h->pidx,
            &h->leaf_cnt, &h->leaf_bin, &h->nfirst, &h->nitem, &h->naxis,
            &h->stats, &h->d_grids, &h->d_cnt_off, &h->roots, &h->scan_bsum,
            &h->scan_side, &h->deep_part};
}

// reinit_device with every per-call buffer taken from the device's scratch:
// the handle's own buffers are set aside for the call and put back after it,
// and the interface, nearest indices and normals of the call are not kept.
int reinit_noalloc(ft_ctx* c, double* d_phi, double* d_phi_ifn, const ft_opts* o, ft_counts* counts,
                   hipStream_t s)
{
    FT_TRY(validate_opts(o));
    if (o->want_nearest || o->want_normals)
        return ft::set_error(FT_ERR_ARG, "ft_reinit_device_noalloc keeps no nearest indices or normals "
                                         "(they would live in the shared scratch)");
    void* base = nullptr;
    FT_TRY(scratch_address(c->device, &base));
    DevBuf saved[64];
    const std::vector<DevBuf*> bufs = call_buffers(c);
    if (bufs.size() > 64) return ft::set_error(FT_ERR_STATE, "too many call buffers");
    for (size_t i = 0; i < bufs.size(); i++) { saved[i] = *bufs[i]; *bufs[i] = DevBuf{}; }
    const uint64_t idx_layout = c->idx_layout;
    const float idx_bs = c->idx_bin_scale, idx_reach = c->idx_reach;
    const int64_t idx_G = c->idx_G;
    int64_t idx_words[kLevels];
    std::copy(c->idx_words, c->idx_words + kLevels, idx_words);
    const int idx_top = c->idx_top;
    c->idx_layout = ~0ull;                           // grids are uploaded into the scratch
    Arena arena;
    arena.base = static_cast<char*>(base);
    arena.size = kScratchBytes;
    t_arena = &arena;
    const int rc = reinit_device(c, d_phi, d_phi_ifn, o, counts, s, false);
    t_arena = nullptr;
    // a call stopped part way (e.g. out of scratch) leaves kernels in flight
    // that write into the scratch: let them end before returning
    const hipError_t es = hipStreamSynchronize(s);
    for (size_t i = 0; i < bufs.size(); i++) *bufs[i] = saved[i];
    c->idx_layout = idx_layout;
    c->idx_bin_scale = idx_bs;
    c->idx_reach = idx_reach;
    c->idx_G = idx_G;
    std::copy(idx_words, idx_words + kLevels, c->idx_words);
    c->idx_top = idx_top;
    c->have_interface = c->have_nearest = c->have_normals = false;
    // Every buffer a reinit sizes must be in call_buffers; one that is not
    // would keep pointing into the shared scratch after the call.  Such a
    // buffer is dropped (not freed) and the call reports it.
    const char* lo = static_cast<const char*>(base);
    bool escaped = false;
    for (DevBuf* b : all_buffers(c)) {
        const char* p = static_cast<const char*>(b->p);
        if (p && p >= lo && p < lo + kScratchBytes) {
            *b = DevBuf{};
            escaped = true;
        }
    }
    if (escaped) return ft::set_error(FT_ERR_INTERNAL, "a per-call buffer was left in the noalloc scratch");
    if (rc == FT_OK && es != hipSuccess)
        return ft::set_error(FT_ERR_HIP, "hipStreamSynchronize failed: %s", hipGetErrorString(es));
    return rc;
}

}  // namespace

// ============================================================================
// C ABI
// ============================================================================
extern "C" {

void ft_opts_default(ft_opts* o)
{
    if (!o) return;
    std::memset(o, 0, sizeof *o);
    o->mode = FT_DIST_POINTS;
    o->blend = FT_BLEND_INIT;
    o->w_phi = 0.75;
    o->w_ifn = 0.25;
    o->band = 0.0;
    o->bin_scale = 0.0f;
    o->want_nearest = 0;
}

const char* ft_last_error(void) { return ft::error_slot().c_str(); }

int ft_device_count(int32_t* n)
{
    if (!n) return ft::set_error(FT_ERR_ARG, "null output");
    int c = 0;
    hipError_t e = hipGetDeviceCount(&c);
    *n = (e == hipSuccess) ? c : 0;
    return FT_OK;
}

int ft_create(int32_t device, ft_handle* out)
{
    if (!out) return ft::set_error(FT_ERR_ARG, "null output");
    *out = nullptr;
    std::lock_guard<std::mutex> lk(g_create_mu);
    int nd = 0;
    if (hipGetDeviceCount(&nd) != hipSuccess || nd <= 0)
        return ft::set_error(FT_ERR_NODEVICE, "no HIP device");
    if (device < 0 || device >= nd) return ft::set_error(FT_ERR_ARG, "device %d out of range", device);
    FT_HIP(hipSetDevice(device));
    ft_ctx* c = new ft_ctx();
    c->device = device;
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess && cus > 0)
        c->cu_count = cus;
    // A blocking stream: a call that passes no stream (NULL, which is also
    // the address of the null stream) runs on this one, and it must still see
    // the caller's work on the null stream before it (a copy into phi) and
    // come before the caller's null-stream work after it.
    if (hipStreamCreateWithFlags(&c->stream, hipStreamDefault) != hipSuccess) {
        delete c;
        return ft::set_error(FT_ERR_HIP, "hipStreamCreate failed");
    }
    // the side stream is ordered by events alone (default priority, as the other)
    if (hipStreamCreateWithFlags(&c->side, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&c->side_fork_ev, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&c->side_join_ev, hipEventDisableTiming) != hipSuccess) {
        if (c->side_fork_ev) (void)hipEventDestroy(c->side_fork_ev);
        if (c->side) (void)hipStreamDestroy(c->side);
        (void)hipStreamDestroy(c->stream);
        delete c;
        return ft::set_error(FT_ERR_HIP, "side stream set-up failed");
    }
    if (ensure(c->scalars, 8 * S_N) != FT_OK ||
        hipHostMalloc((void**)&c->h_scalars, 8 * S_TOP, hipHostMallocDefault) != hipSuccess) {
        (void)hipStreamDestroy(c->stream);
        (void)hipStreamDestroy(c->side);
        (void)hipEventDestroy(c->side_fork_ev);
        (void)hipEventDestroy(c->side_join_ev);
        release(c->scalars);
        delete c;
        return ft::set_error(FT_ERR_NOMEM, "scalar buffers");
    }
    *out = c;
    return FT_OK;
}

int ft_destroy(ft_handle h)
{
    if (!h) return FT_OK;
    (void)hipSetDevice(h->device);
    (void)hipStreamSynchronize(h->side);
    (void)hipStreamSynchronize(h->stream);
    drop_graph(h);
    for (DevBuf* b : all_buffers(h)) release(*b);
    if (h->h_scalars) (void)hipHostFree(h->h_scalars);
    if (h->h_bcg) (void)hipHostFree(h->h_bcg);
    for (hipEvent_t ev : h->bcg_ev)
        if (ev) (void)hipEventDestroy(ev);
    for (int k = 0; k < 2; k++) {
        if (h->stage[k]) (void)hipHostFree(h->stage[k]);
        if (h->stage_ev[k]) (void)hipEventDestroy(h->stage_ev[k]);
    }
    for (int k = 0; k < 5; k++)
        if (h->ev[k]) (void)hipEventDestroy(h->ev[k]);
    (void)hipEventDestroy(h->side_fork_ev);
    (void)hipEventDestroy(h->side_join_ev);
    (void)hipStreamDestroy(h->side);
    (void)hipStreamDestroy(h->stream);
    delete h;
    return FT_OK;
}

int ft_set_nodes(ft_handle h, const float* xyz, int64_t n_nodes)
{
    FT_TRY(check_handle(h));
    if (n_nodes < 0 || n_nodes > INT32_MAX || (n_nodes > 0 && !xyz))
        return ft::set_error(FT_ERR_ARG, "ft_set_nodes: bad arguments");
    h->has_conn = false;
    h->have_interface = false;
    const int64_t no[2] = {0, n_nodes}, zo[2] = {0, 0};
    FT_TRY(set_fields(h, 1, no, zo, zo));
    FT_TRY(ensure(h->xyz, sizeof(float) * 3 * std::max<int64_t>(1, n_nodes)));
    if (n_nodes > 0)
        FT_HIP(hipMemcpyAsync(h->xyz.p, xyz, sizeof(float) * 3 * n_nodes, hipMemcpyHostToDevice, h->stream));
    boxes_from_host(h, xyz);
    return sort_nodes(h);
}

int ft_set_mesh_batch(ft_handle h, int32_t n_fields, const int64_t* node_off, const float* xyz,
                      const int64_t* tet_off, const int32_t* tets, const int64_t* edge_off,
                      const int32_t* edges, const int32_t* t2e)
{
    FT_TRY(check_handle(h));
    if (n_fields < 1 || !node_off || !tet_off || !edge_off || !xyz)
        return ft::set_error(FT_ERR_ARG, "ft_set_mesh_batch: bad arguments");
    if (node_off[0] != 0 || tet_off[0] != 0 || edge_off[0] != 0)
        return ft::set_error(FT_ERR_ARG, "ft_set_mesh_batch: offsets must start at 0");
    for (int k = 0; k < n_fields; k++)
        if (node_off[k + 1] <= node_off[k] || tet_off[k + 1] < tet_off[k] || edge_off[k + 1] < edge_off[k])
            return ft::set_error(FT_ERR_ARG, "ft_set_mesh_batch: field %d has bad offsets", k);
    const int64_t N = node_off[n_fields], T = tet_off[n_fields], E = edge_off[n_fields];
    if (N > INT32_MAX || T > INT32_MAX || E > INT32_MAX)
        return ft::set_error(FT_ERR_ARG, "ft_set_mesh_batch: sizes exceed int32 indices");
    if ((T > 0 && (!tets || !t2e)) || (E > 0 && !edges))
        return ft::set_error(FT_ERR_ARG, "ft_set_mesh_batch: null connectivity");
    // Field-local indices are validated here so that no kernel reads out of bounds.
    for (int k = 0; k < n_fields; k++) {
        const int64_t nk = node_off[k + 1] - node_off[k], ek = edge_off[k + 1] - edge_off[k];
        for (int64_t i = 4 * tet_off[k]; i < 4 * tet_off[k + 1]; i++)
            if (tets[i] < 0 || tets[i] >= nk)
                return ft::set_error(FT_ERR_ARG, "tet %lld (field %d) has node %d out of range",
                                     (long long)(i / 4), k, tets[i]);
        for (int64_t i = 2 * edge_off[k]; i < 2 * edge_off[k + 1]; i++)
            if (edges[i] < 0 || edges[i] >= nk)
                return ft::set_error(FT_ERR_ARG, "edge %lld (field %d) has node %d out of range",
                                     (long long)(i / 2), k, edges[i]);
        for (int64_t i = 6 * tet_off[k]; i < 6 * tet_off[k + 1]; i++)
            if (t2e[i] < 0 || t2e[i] >= ek)
                return ft::set_error(FT_ERR_ARG, "t2e of tet %lld (field %d) has edge %d out of range",
                                     (long long)(i / 6), k, t2e[i]);
    }
    h->has_conn = false;
    h->have_interface = false;
    FT_TRY(set_fields(h, n_fields, node_off, tet_off, edge_off));
    hipStream_t s = h->stream;
    FT_TRY(ensure(h->xyz, sizeof(float) * 3 * N));
    FT_TRY(ensure(h->tets, 16 * std::max<int64_t>(1, T)));
    FT_TRY(ensure(h->edges, 8 * std::max<int64_t>(1, E)));
    FT_TRY(ensure(h->t2e, 24 * std::max<int64_t>(1, T)));
    FT_HIP(hipMemcpyAsync(h->xyz.p, xyz, sizeof(float) * 3 * N, hipMemcpyHostToDevice, s));
    if (T > 0) {
        FT_HIP(hipMemcpyAsync(h->tets.p, tets, 16 * T, hipMemcpyHostToDevice, s));
        FT_HIP(hipMemcpyAsync(h->t2e.p, t2e, 24 * T, hipMemcpyHostToDevice, s));
    }
    if (E > 0) FT_HIP(hipMemcpyAsync(h->edges.p, edges, 8 * E, hipMemcpyHostToDevice, s));
    // field-local -> global indices, in place
    for (int k = 0; k < n_fields; k++) {
        const int64_t nt = tet_off[k + 1] - tet_off[k], ne = edge_off[k + 1] - edge_off[k];
        if (node_off[k] != 0) {
            int32_t* tp = h->tets.as<int32_t>() + 4 * tet_off[k];
            int32_t* ep = h->edges.as<int32_t>() + 2 * edge_off[k];
            if (nt) hipLaunchKernelGGL(k_add_offset, dim3(grid1d(4 * nt)), dim3(kBS), 0, s, tp, 4 * nt, node_off[k], tp);
            if (ne) hipLaunchKernelGGL(k_add_offset, dim3(grid1d(2 * ne)), dim3(kBS), 0, s, ep, 2 * ne, node_off[k], ep);
        }
        if (edge_off[k] != 0 && nt) {
            int32_t* qp = h->t2e.as<int32_t>() + 6 * tet_off[k];
            hipLaunchKernelGGL(k_add_offset, dim3(grid1d(6 * nt)), dim3(kBS), 0, s, qp, 6 * nt, edge_off[k], qp);
        }
    }
    FT_TRY(check_launch());
    boxes_from_host(h, xyz);
    FT_TRY(sort_nodes(h));
    h->has_conn = true;
    return FT_OK;
}

int ft_set_mesh(ft_handle h, const float* xyz, int64_t n_nodes, const int32_t* tets,
                int64_t n_tets, const int32_t* edges, int64_t n_edges, const int32_t* t2e)
{
    FT_TRY(check_handle(h));
    if (n_nodes <= 0 || n_tets < 0 || n_edges < 0)
        return ft::set_error(FT_ERR_ARG, "ft_set_mesh: bad arguments");
    const int64_t no[2] = {0, n_nodes}, to[2] = {0, n_tets}, eo[2] = {0, n_edges};
    return ft_set_mesh_batch(h, 1, no, xyz, to, tets, eo, edges, t2e);
}

int ft_set_kuhn_batch(ft_handle h, int32_t n_fields, const int32_t* dims, const double* origins,
                      const double* spacings, double jitter, uint64_t seed)
{
    FT_TRY(check_handle(h));
    if (n_fields < 1 || !dims || !(jitter >= 0.0 && jitter < 0.5))
        return ft::set_error(FT_ERR_ARG, "ft_set_kuhn_batch: bad arguments");
    std::vector<int64_t> no(n_fields + 1, 0), to(n_fields + 1, 0), eo(n_fields + 1, 0);
    for (int k = 0; k < n_fields; k++) {
        int64_t nn, nt, ne;
        FT_TRY(ft_kuhn_counts(dims[3 * k], dims[3 * k + 1], dims[3 * k + 2], &nn, &nt, &ne));
        no[k + 1] = no[k] + nn;
        to[k + 1] = to[k] + nt;
        eo[k + 1] = eo[k] + ne;
    }
    if (no[n_fields] > INT32_MAX || to[n_fields] > INT32_MAX || eo[n_fields] > INT32_MAX)
        return ft::set_error(FT_ERR_ARG, "ft_set_kuhn_batch: batch exceeds int32 indices");
    h->has_conn = false;
    h->have_interface = false;
    FT_TRY(set_fields(h, n_fields, no.data(), to.data(), eo.data()));
    hipStream_t s = h->stream;
    FT_TRY(ensure(h->xyz, sizeof(float) * 3 * no[n_fields]));
    FT_TRY(ensure(h->tets, 16 * std::max<int64_t>(1, to[n_fields])));
    FT_TRY(ensure(h->edges, 8 * std::max<int64_t>(1, eo[n_fields])));
    FT_TRY(ensure(h->t2e, 24 * std::max<int64_t>(1, to[n_fields])));
    for (int k = 0; k < n_fields; k++) {
        KuhnField f{};
        f.nx = dims[3 * k]; f.ny = dims[3 * k + 1]; f.nz = dims[3 * k + 2];
        const double sp = 1.0 / (std::max(f.nx, std::max(f.ny, f.nz)) - 1);
        for (int q = 0; q < 3; q++) {
            f.origin[q] = origins ? origins[3 * k + q] : 0.0;
            f.spacing[q] = spacings ? spacings[k] : sp;
        }
        f.jitter = jitter;
        f.seed = seed;
        f.node_off = no[k]; f.tet_off = to[k]; f.edge_off = eo[k];
        const int64_t nn = no[k + 1] - no[k], nt = to[k + 1] - to[k];
        hipLaunchKernelGGL(k_kuhn_nodes, dim3(grid1d(nn)), dim3(kBS), 0, s, f, h->xyz.as<float>());
        hipLaunchKernelGGL(k_kuhn_edges, dim3(grid1d(nn)), dim3(kBS), 0, s, f, h->edges.as<int2>());
        hipLaunchKernelGGL(k_kuhn_tets, dim3(grid1d(nt)), dim3(kBS), 0, s, f, h->tets.as<int4>(),
                           h->t2e.as<int32_t>());
        // box: the grid's extent (jitter moves interior nodes only)
        FieldHost& fb = h->fh[k];
        const int d3[3] = {f.nx, f.ny, f.nz};
        for (int q = 0; q < 3; q++) {
            fb.lo[q] = (float)f.origin[q];
            fb.hi[q] = (float)(f.origin[q] + (d3[q] - 1) * f.spacing[q]);
        }
        finish_field_box(fb, nn);
    }
    h->h_est = h->fh[0].h;
    FT_TRY(check_launch());
    FT_TRY(sort_nodes(h));
    h->has_conn = true;
    return FT_OK;
}

int ft_batch_info(ft_handle h, int32_t* n_fields, int64_t* node_off, int64_t* tet_off,
                  int64_t* edge_off)
{
    FT_TRY(check_handle(h));
    if (n_fields) *n_fields = h->nf;
    for (int k = 0; k <= h->nf; k++) {
        if (node_off) node_off[k] = h->node_off[k];
        if (tet_off) tet_off[k] = h->tet_off[k];
        if (edge_off) edge_off[k] = h->edge_off[k];
    }
    return FT_OK;
}

int ft_get_mesh(ft_handle h, float* xyz, int32_t* tets, int32_t* edges, int32_t* t2e)
{
    FT_TRY(check_handle(h));
    if (tets || edges || t2e) FT_TRY(materialize_conn(h));
    hipStream_t s = h->stream;
    if (xyz && h->N) FT_HIP(hipMemcpyAsync(xyz, h->xyz.p, 12 * h->N, hipMemcpyDeviceToHost, s));
    if (tets && h->T) FT_HIP(hipMemcpyAsync(tets, h->tets.p, 16 * h->T, hipMemcpyDeviceToHost, s));
    if (edges && h->E) FT_HIP(hipMemcpyAsync(edges, h->edges.p, 8 * h->E, hipMemcpyDeviceToHost, s));
    if (t2e && h->T) FT_HIP(hipMemcpyAsync(t2e, h->t2e.p, 24 * h->T, hipMemcpyDeviceToHost, s));
    FT_HIP(hipStreamSynchronize(s));
    return FT_OK;
}

// ---- resident meshes --------------------------------------------------------
// A resident mesh is a one-field handle kept only for its mesh and its query
// slots.  A batch of resident meshes reads their tets, t2e and edges in place
// and copies only their node coordinates and slots; it holds a reference to
// each, so a mesh released while a batch still refers to it is freed when
// that batch moves on (its id is free at once).
}  // extern "C" (the registry below is C++)

namespace {
// Ids of released meshes are reused; the serial is not (it grows with every
// mesh created in the process), so (id, serial) names one mesh for good.
struct Resident {
    std::shared_ptr<ft_ctx> c;
    int64_t bytes = 0;
    uint64_t serial = 0;
};
std::mutex g_res_mu;
std::vector<Resident> g_res;
uint64_t g_res_serial = 0;

int resident_finish(ft_ctx* c, int32_t* id)
{
    // drop the set-up workspaces, keep mesh + slots
    DevBuf* tmp[] = {&c->bin_count, &c->bin_prefix, &c->pcode, &c->scan_bsum};
    for (DevBuf* b : tmp) release(*b);
    Resident r;
    r.c = std::shared_ptr<ft_ctx>(c, [](ft_ctx* p) { ft_destroy(p); });
    r.bytes = (int64_t)(c->xyz.cap + c->tets.cap + c->edges.cap + c->t2e.cap + c->perm.cap + c->sx.cap +
                        c->sy.cap + c->sz.cap + c->tile_field.cap + c->tile_sched.cap);
    std::lock_guard<std::mutex> lk(g_res_mu);
    r.serial = ++g_res_serial;
    for (size_t i = 0; i < g_res.size(); i++)
        if (!g_res[i].c) { g_res[i] = r; *id = (int32_t)i; return FT_OK; }
    g_res.push_back(r);
    *id = (int32_t)g_res.size() - 1;
    return FT_OK;
}

std::shared_ptr<ft_ctx> resident_get(int32_t id, uint64_t* serial = nullptr)
{
    std::lock_guard<std::mutex> lk(g_res_mu);
    if (id < 0 || id >= (int32_t)g_res.size()) return nullptr;
    if (serial) *serial = g_res[id].serial;
    return g_res[id].c;
}
}  // namespace

extern "C" {

int ft_mesh_create_kuhn(int32_t device, int32_t nx, int32_t ny, int32_t nz, double jitter,
                        uint64_t seed, int32_t* id)
{
    if (!id) return ft::set_error(FT_ERR_ARG, "null output");
    ft_handle h = nullptr;
    FT_TRY(ft_create(device, &h));
    const int32_t dims[3] = {nx, ny, nz};
    int rc = ft_set_kuhn_batch(h, 1, dims, nullptr, nullptr, jitter, seed);
    if (rc) { ft_destroy(h); return rc; }
    return resident_finish(h, id);
}

int ft_mesh_create(int32_t device, const float* xyz, int64_t n_nodes, const int32_t* tets,
                   int64_t n_tets, const int32_t* edges, int64_t n_edges, const int32_t* t2e,
                   int32_t* id)
{
    if (!id) return ft::set_error(FT_ERR_ARG, "null output");
    ft_handle h = nullptr;
    FT_TRY(ft_create(device, &h));
    int rc = ft_set_mesh(h, xyz, n_nodes, tets, n_tets, edges, n_edges, t2e);
    if (rc) { ft_destroy(h); return rc; }
    return resident_finish(h, id);
}

int ft_mesh_info(int32_t id, int64_t* n_nodes, int64_t* n_tets, int64_t* n_edges, int64_t* bytes)
{
    std::lock_guard<std::mutex> lk(g_res_mu);
    if (id < 0 || id >= (int32_t)g_res.size() || !g_res[id].c)
        return ft::set_error(FT_ERR_ARG, "no resident mesh %d", id);
    const ft_ctx* c = g_res[id].c.get();
    if (n_nodes) *n_nodes = c->N;
    if (n_tets) *n_tets = c->T;
    if (n_edges) *n_edges = c->E;
    if (bytes) *bytes = g_res[id].bytes;
    return FT_OK;
}

int ft_mesh_release(int32_t id)
{
    std::shared_ptr<ft_ctx> c;
    {
        std::lock_guard<std::mutex> lk(g_res_mu);
        if (id < 0 || id >= (int32_t)g_res.size() || !g_res[id].c)
            return ft::set_error(FT_ERR_ARG, "no resident mesh %d", id);
        c.swap(g_res[id].c);
        g_res[id] = Resident{};
    }
    return FT_OK;                     // destroyed here unless a batch still refers to it
}

int ft_set_batch_meshes(ft_handle h, int32_t n_fields, const int32_t* mesh_ids)
{
    FT_TRY(check_handle(h));
    if (n_fields < 1 || !mesh_ids) return ft::set_error(FT_ERR_ARG, "ft_set_batch_meshes: bad arguments");
    std::vector<std::shared_ptr<ft_ctx>> ms(n_fields);
    std::vector<uint64_t> serials(n_fields);
    for (int k = 0; k < n_fields; k++) {
        ms[k] = resident_get(mesh_ids[k], &serials[k]);
        if (!ms[k]) return ft::set_error(FT_ERR_ARG, "no resident mesh %d", mesh_ids[k]);
        if (ms[k]->device != h->device)
            return ft::set_error(FT_ERR_ARG, "resident mesh %d lives on another device", mesh_ids[k]);
    }
    // already set from these very meshes: an id alone is not enough, a
    // released id may since name a new mesh of other dimensions
    if (h->has_conn && h->batch_meshes == serials) return FT_OK;
    std::vector<int64_t> no(n_fields + 1, 0), to(n_fields + 1, 0), eo(n_fields + 1, 0);
    for (int k = 0; k < n_fields; k++) {
        no[k + 1] = no[k] + ms[k]->N;
        to[k + 1] = to[k] + ms[k]->T;
        eo[k + 1] = eo[k] + ms[k]->E;
    }
    if (no[n_fields] > INT32_MAX || to[n_fields] > INT32_MAX || eo[n_fields] > INT32_MAX)
        return ft::set_error(FT_ERR_ARG, "batch exceeds int32 indices");
    h->has_conn = false;
    h->have_interface = false;
    FT_TRY(set_fields(h, n_fields, no.data(), to.data(), eo.data()));
    hipStream_t s = h->stream;
    FT_TRY(ensure(h->xyz, 12 * no[n_fields]));
    std::vector<int64_t> slots(n_fields);
    for (int k = 0; k < n_fields; k++) slots[k] = ms[k]->n_slots;
    FT_TRY(set_slots(h, slots));
    // per-field connectivity pointers: tets, t2e, edges of each mesh
    std::vector<const void*> tab(3 * (size_t)n_fields);
    for (int k = 0; k < n_fields; k++) {
        tab[k] = ms[k]->tets.p;
        tab[n_fields + k] = ms[k]->t2e.p;
        tab[2 * n_fields + k] = ms[k]->edges.p;
    }
    FT_TRY(ensure(h->field_tab, sizeof(void*) * tab.size()));
    FT_HIP(hipMemcpyAsync(h->field_tab.p, tab.data(), sizeof(void*) * tab.size(), hipMemcpyHostToDevice, s));
    FT_TRY(gather_meshes(h, ms, s, false));
    for (int k = 0; k < n_fields; k++) h->fh[k] = ms[k]->fh[0];
    h->h_est = h->fh[0].h;
    FT_HIP(hipStreamSynchronize(s));
    h->field_meshes = std::move(ms);
    h->virt = true;
    h->batch_meshes = serials;
    h->has_conn = true;
    return FT_OK;
}

int ft_get_field_counts(ft_handle h, ft_counts* per_field)
{
    FT_TRY(check_handle(h));
    if (!per_field) return ft::set_error(FT_ERR_ARG, "null output");
    for (int k = 0; k < h->nf; k++)
        per_field[k] = k < (int)h->field_counts.size() ? h->field_counts[k] : ft_counts{};
    return FT_OK;
}

int ft_reinit_batch(ft_handle h, double* d_phi, double* d_phi_ifn, const ft_opts* o,
                    ft_counts* per_field, void* stream)
{
    FT_TRY(check_handle(h));
    hipStream_t s = stream ? (hipStream_t)stream : h->stream;
    ft_counts tot{};
    const int rc = reinit_device(h, d_phi, d_phi_ifn, o, &tot, s);
    if (per_field)
        for (int k = 0; k < h->nf && k < (int)h->field_counts.size(); k++) per_field[k] = h->field_counts[k];
    return rc;
}

int ft_reinit_graph(ft_handle h, double* d_phi, double* d_phi_ifn, const ft_opts* o,
                    ft_counts* per_field, void* stream)
{
    FT_TRY(check_handle(h));
    hipStream_t s = stream ? (hipStream_t)stream : h->stream;
    ft_counts tot{};
    const int rc = reinit_graph(h, d_phi, d_phi_ifn, o, &tot, s);
    if (per_field)
        for (int k = 0; k < h->nf && k < (int)h->field_counts.size(); k++) per_field[k] = h->field_counts[k];
    return rc;
}

int ft_get_counts(ft_handle h, ft_counts* total)
{
    FT_TRY(check_handle(h));
    if (!total) return ft::set_error(FT_ERR_ARG, "null output");
    if (!h->have_interface) return ft::set_error(FT_ERR_STATE, "no interface: reinit first");
    *total = h->last;
    return FT_OK;
}

int ft_get_normals(ft_handle h, float* normals)
{
    FT_TRY(check_handle(h));
    if (!normals) return ft::set_error(FT_ERR_ARG, "null output");
    if (!h->have_normals) return ft::set_error(FT_ERR_STATE, "no normals: reinit with want_normals first");
    if (h->N > 0) FT_HIP(hipMemcpyAsync(normals, h->normals.p, 12 * h->N, hipMemcpyDeviceToHost, h->stream));
    FT_HIP(hipStreamSynchronize(h->stream));
    return FT_OK;
}

int ft_normals_device(ft_handle h, const float** normals)
{
    FT_TRY(check_handle(h));
    if (!normals) return ft::set_error(FT_ERR_ARG, "null output");
    if (!h->have_normals) return ft::set_error(FT_ERR_STATE, "no normals: reinit with want_normals first");
    *normals = h->normals.as<float>();
    return FT_OK;
}

// LevelSet::getInterfaceCurvature (LevelSet.cpp:215-253) of the last reinit
// into the handle's k_if, on stream s.
int enqueue_curvature(ft_ctx* h, hipStream_t s)
{
    FT_TRY(materialize_conn(h));
    if (!h->have_normals || !h->have_interface || !h->last_phi)
        return ft::set_error(FT_ERR_STATE, "curvature needs a reinit with want_normals first");
    const int64_t N = h->N, T = h->T, P = h->last.n_ifp;
    FT_TRY(ensure(h->gsplit, 16 * at_least1(N)));
    FT_TRY(ensure(h->kmesh, 4 * at_least1(N)));
    FT_TRY(ensure(h->k_if, 4 * at_least1(P)));
    if (N > 0) {
        float4* unit = h->gsplit.as<float4>();
        const uint64_t* sc = h->scalars.as<uint64_t>();
        hipLaunchKernelGGL(k_unit_split, dim3(grid1d(N)), dim3(kBS), 0, s, h->normals.as<float>(), N, unit);
        if (T > 0)
            hipLaunchKernelGGL(k_tet_grad_diag, dim3(grid1d(T)), dim3(kBS), 0, s, h->tets.as<int4>(), T,
                               h->xyz.as<float>(), unit, h->grad_t.as<float4>(), sc);
        hipLaunchKernelGGL(k_node_div, dim3(grid1d(N)), dim3(kBS), 0, s, h->n2t_off.as<uint64_t>(),
                           h->n2t_ids.as<int32_t>(), h->grad_t.as<float4>(), N, h->kmesh.as<float>());
        if (P > 0)
            hipLaunchKernelGGL(k_curv_points, dim3(grid1d(P)), dim3(kBS), 0, s, h->ifp2e.as<int32_t>(), P,
                               h->edges.as<int2>(), h->last_phi, h->kmesh.as<float>(), h->k_if.as<float>());
        FT_TRY(check_launch());
    }
    return FT_OK;
}

int ft_interface_curvature(ft_handle h, float* k_if, void* stream)
{
    FT_TRY(check_handle(h));
    if (!k_if) return ft::set_error(FT_ERR_ARG, "null output");
    hipStream_t s = stream ? (hipStream_t)stream : h->stream;
    FT_TRY(enqueue_curvature(h, s));
    const int64_t P = h->last.n_ifp;
    if (P > 0) FT_HIP(hipMemcpyAsync(k_if, h->k_if.p, 4 * P, hipMemcpyDeviceToHost, s));
    FT_HIP(hipStreamSynchronize(s));
    return FT_OK;
}

// Flow::surfaceTension_ (src/growth/Flow.cpp:307-341) on device arrays.
int surface_tension(ft_ctx* h, float st, int32_t rho, double* fx, double* fy, double* fz, hipStream_t s)
{
    FT_TRY(materialize_conn(h));
    FT_TRY(enqueue_curvature(h, s));
    const int64_t N = h->N, P = h->last.n_ifp;
    if (N == 0 || P == 0) return FT_OK;
    FT_TRY(ensure(h->st_cnt, 4 * N));
    FT_TRY(ensure(h->st_off, 8 * (N + 1)));
    FT_TRY(ensure(h->st_ids, 4 * 2 * P));
    uint32_t* cnt = h->st_cnt.as<uint32_t>();
    uint64_t* off = h->st_off.as<uint64_t>();
    int32_t* ids = h->st_ids.as<int32_t>();
    const int32_t* ifp2e = h->ifp2e.as<int32_t>();
    const int2* edges = h->edges.as<int2>();
    FT_TRY(fill<uint32_t>(s, cnt, N, 0u));
    hipLaunchKernelGGL(k_st_count, dim3(grid1d(P)), dim3(kBS), 0, s, ifp2e, P, edges, cnt);
    FT_TRY(scan<uint32_t, uint64_t>(h, s, cnt, off, N, off + N, LoadClear{}));   // cnt: then the fill's cursors
    hipLaunchKernelGGL(k_st_fill, dim3(grid1d(P)), dim3(kBS), 0, s, ifp2e, P, edges, off, cnt, ids);
    hipLaunchKernelGGL(k_n2t_sort, dim3(grid1d(N)), dim3(kBS), 0, s, off, N, ids);
    hipLaunchKernelGGL(k_st_apply, dim3(grid1d(N)), dim3(kBS), 0, s, off, ids, N, ifp2e, edges,
                       h->last_phi, h->k_if.as<float>(), h->ifp_area.as<float>(), h->normals.as<float>(),
                       st, rho, fx, fy, fz);
    FT_TRY(check_launch());
    return FT_OK;
}

int ft_surface_tension_device(ft_handle h, float st, int32_t rho, double* fx, double* fy, double* fz,
                              void* stream)
{
    FT_TRY(check_handle(h));
    if (h->N > 0 && (!fx || !fy || !fz)) return ft::set_error(FT_ERR_ARG, "null force array");
    hipStream_t s = stream ? (hipStream_t)stream : h->stream;
    FT_TRY(surface_tension(h, st, rho, fx, fy, fz, s));
    FT_HIP(hipStreamSynchronize(s));
    return FT_OK;
}

int ft_surface_tension(ft_handle h, float st, int32_t rho, double* fx, double* fy, double* fz)
{
    FT_TRY(check_handle(h));
    const int64_t N = h->N;
    if (N > 0 && (!fx || !fy || !fz)) return ft::set_error(FT_ERR_ARG, "null force array");
    hipStream_t s = h->stream;
    FT_TRY(ensure(h->st_f, 24 * at_least1(N)));
    double* d = h->st_f.as<double>();
    double* host[3] = {fx, fy, fz};
    for (int c = 0; c < 3; c++) FT_TRY(copy_h2d(h, d + c * N, host[c], 8 * (size_t)N, s));
    FT_TRY(surface_tension(h, st, rho, d, d + N, d + 2 * N, s));
    return copy_d2h(h, {{fx, d, 8 * (size_t)N}, {fy, d + N, 8 * (size_t)N}, {fz, d + 2 * N, 8 * (size_t)N}}, s);
}

// ---- Advection (LevelSet::update, LevelSet.cpp:89-141) ---------------------
// Quadrature(2, P1) (Quadrature.hpp:23-36) at the float shape functions
// (Tetrahedron.hpp:30-34): the point coordinates go in as float and phi_0 =
// 1.0 - x - y - z comes back rounded to float: at the points (a, b, b),
// (b, a, b), (b, b, a) the same value, at (b, b, b) the float of a.
FemQuad fem_quad()
{
    FemQuad q;
    const double a = (5.0 + 3.0 * std::sqrt(5.0)) / 20.0, b = (5.0 - std::sqrt(5.0)) / 20.0;
    const float ha = (float)a, lb = (float)b;
    q.hi = (double)ha;
    q.lo = (double)lb;
    q.lo0 = (double)(float)(((1.0 - (double)ha) - (double)lb) - (double)lb);
    q.w = 0.25 / 6.0;
    return q;
}

size_t fem_lds(const ft_ctx* h, int form) { return fem_lds_bytes(h->fem_stride, form); }
unsigned fem_grid(int64_t N) { return (unsigned)((N + kFemRowsPerWave - 1) / kFemRowsPerWave); }

FemEll fem_ell(ft_ctx* h)
{
    return FemEll{h->fem_len.as<int32_t>(), h->fem_soff.as<uint64_t>(), h->fem_cols.as<int32_t>(),
                  h->fem_nd.as<int32_t>(), h->fem_diag.as<int32_t>(), h->fem_dmask.as<uint32_t>(), h->tets_twice};
}

// The sliced-ELL pattern and the mass matrix (LevelSet::init,
// LevelSet.cpp:35-39), once per mesh layout.
int fem_setup(ft_ctx* h, hipStream_t s)
{
    FT_TRY(materialize_conn(h));
    if (h->fem_layout == h->layout_gen) return FT_OK;
    if (!h->has_conn) return ft::set_error(FT_ERR_STATE, "advection needs a mesh (ft_set_mesh)");
    FT_TRY(build_node_tets(h, s));
    const int64_t N = h->N, ns = (N + kFemSlice - 1) / kFemSlice;
    FT_TRY(ensure(h->fem_len, 4 * at_least1(N)));
    FT_TRY(ensure(h->fem_w, 4 * at_least1(ns)));
    FT_TRY(ensure(h->fem_soff, 8 * (ns + 1)));
    FT_TRY(ensure(h->fem_flag, 16));
    uint32_t* w = h->fem_w.as<uint32_t>();
    uint64_t* soff = h->fem_soff.as<uint64_t>();
    FT_TRY(fill<unsigned>(s, h->fem_flag.as<unsigned>(), 2, 0u));   // overflow, longest row
    FT_TRY(fill<uint64_t>(s, soff + ns, 1, 0ull));
    if (ns > 0) {
        hipLaunchKernelGGL(k_fem_rowlen, dim3((unsigned)ns), dim3(kFemSlice), 0, s, h->n2t_off.as<uint64_t>(),
                           h->n2t_ids.as<int32_t>(), h->tets.as<int4>(), N, h->fem_len.as<int32_t>(), w,
                           h->fem_flag.as<unsigned>());
        FT_TRY(scan<uint32_t, uint64_t>(h, s, w, soff, ns, soff + ns, LoadSame{}));
    }
    uint64_t total = 0;
    unsigned flag[2] = {0, 0};
    FT_HIP(hipMemcpyAsync(&total, soff + ns, 8, hipMemcpyDeviceToHost, s));
    FT_HIP(hipMemcpyAsync(flag, h->fem_flag.p, 8, hipMemcpyDeviceToHost, s));
    FT_HIP(hipStreamSynchronize(s));
    if (flag[0])
        return ft::set_error(FT_ERR_ARG, "a node shares tets with more than %d nodes", kFemMaxCols - 1);
    const int64_t nnz = (int64_t)total * kFemSlice;
    FT_TRY(ensure(h->fem_cols, 4 * at_least1(nnz)));
    FT_TRY(ensure(h->fem_m, 8 * at_least1(nnz)));
    FT_TRY(ensure(h->fem_l, 8 * at_least1(nnz)));
    FT_TRY(ensure(h->fem_map, 4 * at_least1(4 * h->T)));             // one word per n2t entry
    FT_TRY(ensure(h->fem_nd, 4 * at_least1(ns)));
    FT_TRY(ensure(h->fem_diag, 4 * kFemDiags * at_least1(ns)));
    FT_TRY(ensure(h->fem_dmask, 4 * at_least1(N)));
    h->fem_stride = (int)flag[1] | 1;
    const FemEll e = fem_ell(h);
    if (ns > 0) {
        hipLaunchKernelGGL(k_fem_rowfill, dim3((unsigned)ns), dim3(kFemSlice), 0, s, h->n2t_off.as<uint64_t>(),
                           h->n2t_ids.as<int32_t>(), h->tets.as<int4>(), N, e, w, h->fem_cols.as<int32_t>(),
                           h->fem_map.as<uint32_t>());
        hipLaunchKernelGGL(k_fem_diags, dim3((unsigned)ns), dim3(kFemSlice), 0, s, N, e, h->fem_nd.as<int32_t>(),
                           h->fem_diag.as<int32_t>(), h->fem_dmask.as<uint32_t>());
        hipLaunchKernelGGL(k_fem_mass, dim3(fem_grid(N)), dim3(64), fem_lds(h, 0), s,
                           h->n2t_off.as<uint64_t>(), h->fem_map.as<uint32_t>(), h->xyz.as<float>(), N, fem_quad(), e, h->fem_stride,
                           h->fem_m.as<double>());
    }
    FT_TRY(check_launch());
    FT_HIP(hipStreamSynchronize(s));
    h->fem_nnz = nnz;
    h->fem_layout = h->layout_gen;
    return FT_OK;
}

int bcg_fin(ft_ctx* h, hipStream_t s, int64_t nb, int step, bool read, double tol2 = 0.0, double eps2 = 0.0)
{
    hipLaunchKernelGGL(k_bcg_fin, dim3(1), dim3(256), 0, s, h->bcg_part.as<double>(), nb, step,
                       h->bcg_sc.as<BcgScalars>(), tol2, eps2);
    if (read) {
        FT_HIP(hipMemcpyAsync(h->h_bcg, h->bcg_sc.p, sizeof(BcgScalars), hipMemcpyDeviceToHost, s));
        FT_HIP(hipStreamSynchronize(s));
    }
    return FT_OK;
}

// Crank-Nicolson step of LevelSet::update on device phi (in/out) and flow
// (4 N: velocity x, y, z, pressure), BiCGSTAB to tol in at most max_iters.
int advect(ft_ctx* h, double* d_phi, const double* d_flow, double dt, double tol, int32_t max_iters,
           ft_advect_info* info, hipStream_t s)
{
    *info = ft_advect_info{};
    if (h->nf != 1) return ft::set_error(FT_ERR_STATE, "advection needs a single field");
    if (!h->has_conn) return ft::set_error(FT_ERR_STATE, "advection needs a mesh (ft_set_mesh)");
    const int64_t N = h->N;
    if (dt < FLT_MIN || N == 0) { info->skipped = 1; info->converged = 1; return FT_OK; }   // :92-93
    const int64_t nb = std::min<int64_t>((N + kBcgBS - 1) / kBcgBS, kBcgGrid);
    FT_TRY(ensure(h->bcg_part, 16 * (size_t)nb));
    FT_TRY(ensure(h->bcg_sc, sizeof(BcgScalars)));
    if (!h->h_bcg) FT_HIP(hipHostMalloc(&h->h_bcg, (1 + kBcgAhead) * sizeof(BcgScalars), hipHostMallocDefault));
    for (hipEvent_t& ev : h->bcg_ev)
        if (!ev) FT_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    BcgScalars* hs = static_cast<BcgScalars*>(h->h_bcg);
    double* part = h->bcg_part.as<double>();
    BcgScalars* sc = h->bcg_sc.as<BcgScalars>();
    // flow.norm() < FLT_MIN: nothing to do (:93); NaN velocity: error (:112-115)
    hipLaunchKernelGGL(k_flow_check, dim3((unsigned)nb), dim3(kBcgBS), 0, s, d_flow, N, part);
    FT_TRY(bcg_fin(h, s, nb, BCG_SUMS, true));
    if (std::sqrt(hs->tt) < FLT_MIN) { info->skipped = 1; info->converged = 1; return FT_OK; }
    if (hs->ts > 0.0) return ft::set_error(FT_ERR_ARG, "the velocity has NaN (LevelSet.cpp:112-115)");
    FT_TRY(fem_setup(h, s));
    FT_TRY(ensure(h->bcg_vec, 11 * 8 * (size_t)N));
    double* vec = h->bcg_vec.as<double>();
    double *x = vec, *r = vec + N, *r0 = vec + 2 * N, *p = vec + 3 * N, *v = vec + 4 * N, *t = vec + 5 * N,
           *invdiag = vec + 6 * N, *b = vec + 7 * N, *y = vec + 8 * N, *sv = vec + 9 * N, *z = vec + 10 * N;
    const FemEll e = fem_ell(h);
    double* lv = h->fem_l.as<double>();
    FT_TRY(ensure(h->adv_vel3, 24 * (size_t)N));
    hipLaunchKernelGGL(k_vel_interleave, dim3(grid1d(N)), dim3(kBS), 0, s, d_flow, N, h->adv_vel3.as<double>());
    hipLaunchKernelGGL(k_fem_cn, dim3(fem_grid(N)), dim3(64), fem_lds(h, 1), s, h->n2t_off.as<uint64_t>(),
                       h->fem_map.as<uint32_t>(), h->xyz.as<float>(), h->adv_vel3.as<double>(), N, fem_quad(), e, h->fem_stride,
                       h->fem_m.as<double>(), 0.5 * dt, d_phi, lv, invdiag, b, x, r, r0, p, v);
    hipLaunchKernelGGL(k_dots2, dim3((unsigned)nb), dim3(kBcgBS), 0, s, N, r, r, b, b, part);
    FT_TRY(check_launch());
    FT_TRY(bcg_fin(h, s, nb, BCG_INIT, true));
    const double tol_ = tol > 0.0 ? tol : DBL_EPSILON;                 // Eigen's defaults
    const int64_t max_it = max_iters > 0 ? max_iters : 2 * N;
    if (hs->bb == 0.0) {                                               // zero right-hand side: x = 0
        FT_TRY(fill<double>(s, d_phi, N, 0.0));
        FT_HIP(hipStreamSynchronize(s));
        info->iterations = (int32_t)std::min<int64_t>(max_it, INT32_MAX);
        info->error = tol_;
        info->converged = 1;
        return FT_OK;
    }
    const double tol2 = tol_ * tol_ * hs->bb, eps2 = DBL_EPSILON * DBL_EPSILON;
    int64_t it = 0, restarts = 0;
    const dim3 g((unsigned)nb), bs(kBcgBS);
    // One iteration is enqueued ahead of the one whose scalars are awaited, so
    // that the device does not wait for the host (an update at 72^3 from host
    // arrays 2.70 ms without, 2.59 with, 2.61 with two ahead); the one after
    // the last finds `stop` set and changes nothing.
    BcgScalars cur = *hs;
    int64_t sent = 0, seen = 0;                                        // iterations enqueued, read back
    auto iterate = [&]() -> int {
        hipLaunchKernelGGL(k_bcg_p, g, bs, 0, s, N, sc, r, v, invdiag, p, y);
        hipLaunchKernelGGL(k_bcg_v, g, bs, 0, s, N, sc, e, lv, y, r0, v, part);
        FT_TRY(bcg_fin(h, s, nb, BCG_ALPHA, false));
        hipLaunchKernelGGL(k_bcg_s, g, bs, 0, s, N, sc, invdiag, r, v, sv, z);
        hipLaunchKernelGGL(k_bcg_t, g, bs, 0, s, N, sc, e, lv, z, sv, t, part);
        FT_TRY(bcg_fin(h, s, nb, BCG_W, false));
        hipLaunchKernelGGL(k_bcg_x, g, bs, 0, s, N, y, sv, z, t, r0, sc, x, r, part);
        FT_TRY(bcg_fin(h, s, nb, BCG_END, false, tol2, eps2));
        FT_HIP(hipMemcpyAsync(hs + 1 + sent % kBcgAhead, sc, sizeof(BcgScalars), hipMemcpyDeviceToHost, s));
        FT_HIP(hipEventRecord(h->bcg_ev[sent % kBcgAhead], s));
        sent++;
        return FT_OK;
    };
    while (bcg_goes_on(cur, tol2) && it < max_it) {
        if (bcg_small_rho(cur, eps2)) {
            hipLaunchKernelGGL(k_bcg_restart, g, bs, 0, s, N, e, lv, b, x, r, r0, part);
            FT_TRY(bcg_fin(h, s, nb, BCG_RESTART, false));
            if (restarts++ == 0) it = 0;
        }
        while (sent < seen + kBcgAhead && it + (sent - seen) < max_it) FT_TRY(iterate());
        FT_HIP(hipEventSynchronize(h->bcg_ev[seen % kBcgAhead]));
        cur = hs[1 + seen % kBcgAhead];
        seen = cur.stop ? sent : seen + 1;                             // those after a stop did nothing
        it++;
    }
    FT_TRY(check_launch());
    info->iterations = (int32_t)std::min<int64_t>(it, INT32_MAX);
    info->restarts = (int32_t)restarts;
    info->error = std::sqrt(cur.rr / cur.bb);
    info->converged = info->error <= tol_;
    if (!info->converged) {                                            // :135-139, phi kept
        FT_HIP(hipStreamSynchronize(s));
        return ft::set_error(FT_ERR_SOLVER, "BiCGSTAB stopped at |r|/|b| = %g > %g after %lld iterations",
                             info->error, tol_, (long long)it);
    }
    FT_HIP(hipMemcpyAsync(d_phi, x, 8 * N, hipMemcpyDeviceToDevice, s));
    FT_HIP(hipStreamSynchronize(s));
    return FT_OK;
}

int ft_advect_device(ft_handle h, double* d_phi, const double* d_flow, double dt, double tol,
                     int32_t max_iters, ft_advect_info* info, void* stream)
{
    FT_TRY(check_handle(h));
    if (h->N > 0 && (!d_phi || !d_flow)) return ft::set_error(FT_ERR_ARG, "null phi or flow");
    ft_advect_info tmp;
    return advect(h, d_phi, d_flow, dt, tol, max_iters, info ? info : &tmp,
                  stream ? (hipStream_t)stream : h->stream);
}

int ft_advect(ft_handle h, double* phi, const double* flow, double dt, double tol, int32_t max_iters,
              ft_advect_info* info)
{
    FT_TRY(check_handle(h));
    const int64_t N = h->N;
    if (N > 0 && (!phi || !flow)) return ft::set_error(FT_ERR_ARG, "null phi or flow");
    ft_advect_info tmp;
    if (!info) info = &tmp;
    hipStream_t s = h->stream;
    FT_TRY(ensure(h->adv_phi, 8 * at_least1(N)));
    FT_TRY(ensure(h->adv_flow, 32 * at_least1(N)));
    FT_TRY(copy_h2d(h, h->adv_phi.p, phi, 8 * (size_t)N, s));
    FT_TRY(copy_h2d(h, h->adv_flow.p, flow, 32 * (size_t)N, s));
    FT_TRY(advect(h, h->adv_phi.as<double>(), h->adv_flow.as<double>(), dt, tol, max_iters, info, s));
    if (!info->skipped) FT_TRY(copy_d2h(h, {{phi, h->adv_phi.p, 8 * (size_t)N}}, s));
    return FT_OK;
}

int ft_fem_assemble(ft_handle h, int32_t form, const double* vel, int64_t* row_off, int32_t* cols,
                    double* vals)
{
    FT_TRY(check_handle(h));
    if ((form != 0 && form != 1) || !row_off || (cols && !vals) || (form == 1 && cols && !vel))
        return ft::set_error(FT_ERR_ARG, "ft_fem_assemble: bad arguments");
    if (h->nf != 1) return ft::set_error(FT_ERR_STATE, "needs a single field");
    hipStream_t s = h->stream;
    FT_TRY(fem_setup(h, s));
    const int64_t N = h->N;
    FT_TRY(ensure(h->fem_csr_off, 8 * (N + 1)));
    uint64_t* off = h->fem_csr_off.as<uint64_t>();
    FT_TRY(fill<uint64_t>(s, off + N, 1, 0ull));
    if (N > 0) FT_TRY(scan<int32_t, uint64_t>(h, s, h->fem_len.as<int32_t>(), off, N, off + N, LoadSame{}));
    FT_HIP(hipMemcpyAsync(row_off, off, 8 * (N + 1), hipMemcpyDeviceToHost, s));
    FT_HIP(hipStreamSynchronize(s));
    if (!cols) return FT_OK;                                           // sizes only
    const int64_t nnz = row_off[N];
    const FemEll e = fem_ell(h);
    const double* src = h->fem_m.as<double>();
    if (form == 1) {
        FT_TRY(ensure(h->adv_flow, 32 * at_least1(N)));
        FT_HIP(hipMemcpyAsync(h->adv_flow.p, vel, 24 * N, hipMemcpyHostToDevice, s));
        FT_TRY(ensure(h->adv_vel3, 24 * (size_t)N));
        hipLaunchKernelGGL(k_vel_interleave, dim3(grid1d(N)), dim3(kBS), 0, s, h->adv_flow.as<double>(), N,
                           h->adv_vel3.as<double>());
        hipLaunchKernelGGL(k_fem_adv, dim3(fem_grid(N)), dim3(64), fem_lds(h, 1), s, h->n2t_off.as<uint64_t>(),
                           h->fem_map.as<uint32_t>(), h->xyz.as<float>(), h->adv_vel3.as<double>(), N, fem_quad(), e, h->fem_stride,
                           h->fem_l.as<double>());
        src = h->fem_l.as<double>();
    }
    const int64_t cbytes = (4 * at_least1(nnz) + 255) & ~(int64_t)255;   // CSR staging: cols, vals
    FT_TRY(ensure(h->bcg_vec, cbytes + 8 * at_least1(nnz)));
    int32_t* dc = h->bcg_vec.as<int32_t>();
    double* dv = reinterpret_cast<double*>(h->bcg_vec.as<char>() + cbytes);
    if (N > 0)
        hipLaunchKernelGGL(k_ell_to_csr, dim3(grid1d(N)), dim3(kBS), 0, s, N, e, src, off, dc, dv);
    FT_TRY(check_launch());
    if (nnz > 0) {
        FT_HIP(hipMemcpyAsync(cols, dc, 4 * nnz, hipMemcpyDeviceToHost, s));
        FT_HIP(hipMemcpyAsync(vals, dv, 8 * nnz, hipMemcpyDeviceToHost, s));
    }
    FT_HIP(hipStreamSynchronize(s));
    return FT_OK;
}

int ft_graph_stats(ft_handle h, int64_t* captures, int64_t* launches)
{
    FT_TRY(check_handle(h));
    if (captures) *captures = h->graph.captures;
    if (launches) *launches = h->graph.launches;
    return FT_OK;
}

int ft_reset_phi_points(ft_handle h, const float* ifp, int64_t n_ifp, double* phi_n)
{
    FT_TRY(check_handle(h));
    if (n_ifp < 0 || n_ifp > INT32_MAX || (n_ifp > 0 && !ifp) || (h->N > 0 && !phi_n))
        return ft::set_error(FT_ERR_ARG, "ft_reset_phi_points: bad arguments");
    if (h->nf != 1) return ft::set_error(FT_ERR_STATE, "ft_reset_phi_points needs a single field");
    hipStream_t s = h->stream;
    FT_TRY(ensure(h->phi_tmp, 8 * std::max<int64_t>(1, h->N)));
    FT_TRY(ensure(h->ifp, 12 * std::max<int64_t>(1, n_ifp)));
    FT_TRY(copy_h2d(h, h->ifp.p, ifp, 12 * (size_t)n_ifp, s));
    FT_TRY(copy_h2d(h, h->phi_tmp.p, phi_n, 8 * (size_t)h->N, s));
    h->have_interface = false;
    // the crossing points are given: their count goes where the edge scan
    // would have put it, and the search runs as in a reinit
    Caps cp;
    cp.P = n_ifp;
    SearchSpec sp;
    sp.mode = 0;
    sp.phi_old = h->phi_tmp.as<double>();
    sp.phi_out = h->phi_tmp.as<double>();
    sp.epi = EPI_RAW;
    sp.want_nearest = true;
    uint64_t* sc = h->scalars.as<uint64_t>();
    FT_TRY(index_setup(h, s, 0.0f, sp.mode, far_reach(h->fh[0], ifp, n_ifp)));
    FT_TRY(ensure_stage(h, 0, cp, 0, true));
    WordRanges set;
    set.add(sc + S_BLK, 2, 0u);
    set.add(sc + S_EDGES, 1, (uint32_t)n_ifp);
    set.add(reinterpret_cast<uint32_t*>(sc + S_EDGES) + 1, 1, 0u);
    set.add(sc + S_ERR, 2, ~0u);
    set.add(sc + S_CAP, 2, 0u);
    FT_TRY(set_words(s, set));
    SideJoin join{h, s};
    FT_TRY(enqueue_search(h, s, sp, cp, true, false));
    ft_counts cnt{};
    FT_TRY(collect(h, s, true, &cnt));
    h->have_interface = false;        // points only: no triangles, p2t or areas
    return copy_d2h(h, {{phi_n, h->phi_tmp.p, 8 * (size_t)h->N}}, s);
}

int ft_reinit_device(ft_handle h, double* d_phi, double* d_phi_ifn, const ft_opts* o,
                     ft_counts* counts, void* stream)
{
    FT_TRY(check_handle(h));
    hipStream_t s = stream ? (hipStream_t)stream : h->stream;
    return reinit_device(h, d_phi, d_phi_ifn, o, counts, s);
}

int ft_reinit_device_noalloc(ft_handle h, double* d_phi, double* d_phi_ifn, const ft_opts* o,
                             ft_counts* counts, void* stream)
{
    FT_TRY(check_handle(h));
    if (!d_phi) return ft::set_error(FT_ERR_ARG, "null phi");
    hipStream_t s = stream ? (hipStream_t)stream : h->stream;
    return reinit_noalloc(h, d_phi, d_phi_ifn, o, counts, s);
}

int ft_reinit(ft_handle h, double* phi, double* phi_ifn, const ft_opts* o, ft_counts* counts)
{
    FT_TRY(check_handle(h));
    if (!phi) return ft::set_error(FT_ERR_ARG, "null phi");
    hipStream_t s = h->stream;
    FT_TRY(ensure(h->phi_tmp, 8 * std::max<int64_t>(1, h->N)));
    if (phi_ifn) FT_TRY(ensure(h->phi_ifn_tmp, 8 * std::max<int64_t>(1, h->N)));
    FT_TRY(copy_h2d(h, h->phi_tmp.p, phi, 8 * h->N, s));
    FT_TRY(reinit_device(h, h->phi_tmp.as<double>(), phi_ifn ? h->phi_ifn_tmp.as<double>() : nullptr,
                         o, counts, s));
    std::vector<D2H> out{{phi, h->phi_tmp.p, 8 * (size_t)h->N}};
    if (phi_ifn) out.push_back({phi_ifn, h->phi_ifn_tmp.p, 8 * (size_t)h->N});
    return copy_d2h(h, out, s);
}

int ft_get_interface(ft_handle h, float* ifp, int32_t* ifp2e, int32_t* tris, int32_t* if_elems,
                     float* ifp_area, int32_t* p2t_offsets, int32_t* p2t_tris)
{
    FT_TRY(check_handle(h));
    if (!h->have_interface) return ft::set_error(FT_ERR_STATE, "no interface from a reinit");
    const int64_t P = h->last.n_ifp, F = h->last.n_tri, X = h->last.n_if_elems;
    hipStream_t s = h->stream;
    if (ifp && P) FT_HIP(hipMemcpyAsync(ifp, h->ifp.p, 12 * P, hipMemcpyDeviceToHost, s));
    if (ifp2e && P) FT_HIP(hipMemcpyAsync(ifp2e, h->ifp2e.p, 4 * P, hipMemcpyDeviceToHost, s));
    if (tris && F) FT_HIP(hipMemcpyAsync(tris, h->tris.p, 16 * F, hipMemcpyDeviceToHost, s));
    if (if_elems && X) FT_HIP(hipMemcpyAsync(if_elems, h->if_elems.p, 4 * X, hipMemcpyDeviceToHost, s));
    if (ifp_area && P) FT_HIP(hipMemcpyAsync(ifp_area, h->ifp_area.p, 4 * P, hipMemcpyDeviceToHost, s));
    if (p2t_offsets) FT_HIP(hipMemcpyAsync(p2t_offsets, h->p2t_off.p, 4 * (P + 1), hipMemcpyDeviceToHost, s));
    if (p2t_tris && F) FT_HIP(hipMemcpyAsync(p2t_tris, h->p2t.p, 12 * F, hipMemcpyDeviceToHost, s));
    FT_HIP(hipStreamSynchronize(s));
    return FT_OK;
}

int ft_get_nearest(ft_handle h, int32_t* nearest)
{
    FT_TRY(check_handle(h));
    if (!nearest) return ft::set_error(FT_ERR_ARG, "null output");
    if (!h->have_nearest) return ft::set_error(FT_ERR_STATE, "last call kept no nearest indices");
    FT_HIP(hipMemcpyAsync(nearest, h->nearest.p, 4 * h->N, hipMemcpyDeviceToHost, h->stream));
    FT_HIP(hipStreamSynchronize(h->stream));
    return FT_OK;
}

int ft_set_timing(ft_handle h, int32_t on)
{
    FT_TRY(check_handle(h));
    if (on && !h->ev[0])
        for (int k = 0; k < 5; k++) FT_HIP(hipEventCreate(&h->ev[k]));
    h->timing = on != 0;
    for (int k = 0; k < 4; k++) h->phase_ms[k] = 0.0;
    h->timed_calls = 0;
    return FT_OK;
}

int ft_get_timing(ft_handle h, double* phase_ms, int64_t* calls)
{
    FT_TRY(check_handle(h));
    if (!phase_ms || !calls) return ft::set_error(FT_ERR_ARG, "null output");
    for (int k = 0; k < 4; k++) phase_ms[k] = h->phase_ms[k];
    *calls = h->timed_calls;
    return FT_OK;
}

int ft_interface_device(ft_handle h, const float** ifp, const int32_t** tris, const int32_t** ifp2e)
{
    FT_TRY(check_handle(h));
    if (!h->have_interface) return ft::set_error(FT_ERR_STATE, "no interface from a reinit");
    if (ifp) *ifp = h->ifp.as<float>();
    if (tris) *tris = h->tris.as<int32_t>();
    if (ifp2e) *ifp2e = h->ifp2e.as<int32_t>();
    return FT_OK;
}

}  // extern "C"
