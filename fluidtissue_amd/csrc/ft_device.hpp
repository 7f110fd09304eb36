// ft_device.hpp -- device-side building blocks shared by the reinit kernels:
// bit tests, wave64/block scans, Morton codes and the point/triangle
// distance functions.
#pragma once

#include <hip/hip_runtime.h>
#include <cfloat>
#include <cstdint>

namespace ftd {

constexpr int kWave = 64;

__device__ __forceinline__ int lane_id() { return threadIdx.x & (kWave - 1); }

__device__ __forceinline__ int sign_bit(double x)
{
    return (int)((unsigned long long)__double_as_longlong(x) >> 63);
}

__device__ __forceinline__ int get_bit(const uint64_t* bits, int64_t i)
{
    return (int)((bits[i >> 6] >> (i & 63)) & 1ull);
}

// Load of element i of a read-only array through the constant address space:
// at a wave-uniform address this compiles to scalar (SMEM) loads into SGPRs.
template <class T>
__device__ __forceinline__ T cload(const T* p, int64_t i)
{
    static_assert(sizeof(T) % 4 == 0, "dword-sized records only");
    T v;
    unsigned* d = reinterpret_cast<unsigned*>(&v);
    const __attribute__((address_space(4))) unsigned* src =
        (const __attribute__((address_space(4))) unsigned*)(p + i);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(T) / 4); k++) d[k] = src[k];
    return v;
}

// ---- scans ----------------------------------------------------------------
__device__ __forceinline__ uint64_t shfl_up_u64(uint64_t v, int d, int width = kWave)
{
    const unsigned lo = __shfl_up((unsigned)(v & 0xffffffffu), d, width);
    const unsigned hi = __shfl_up((unsigned)(v >> 32), d, width);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint32_t shfl_up_any(uint32_t v, int d, int width = kWave)
{
    return __shfl_up(v, d, width);
}
__device__ __forceinline__ uint64_t shfl_up_any(uint64_t v, int d, int width = kWave)
{
    return shfl_up_u64(v, d, width);
}

// Five 32-bit counters scanned together (the index's levels): a = primitives
// and level-1 nodes, b = level 2 and level 3, c = level 4; low halves first.
struct Lv {
    uint64_t a, b, c;
    Lv() = default;
    __device__ explicit Lv(int v) : a((uint64_t)v), b((uint64_t)v), c((uint64_t)v) {}
    __device__ Lv& operator+=(const Lv& o) { a += o.a; b += o.b; c += o.c; return *this; }
    __device__ Lv operator+(const Lv& o) const { Lv r = *this; r += o; return r; }
    __device__ Lv operator-(const Lv& o) const { Lv r = *this; r.a -= o.a; r.b -= o.b; r.c -= o.c; return r; }
};
__device__ __forceinline__ Lv shfl_up_any(const Lv& v, int d, int width = kWave)
{
    Lv r;
    r.a = shfl_up_u64(v.a, d, width);
    r.b = shfl_up_u64(v.b, d, width);
    r.c = shfl_up_u64(v.c, d, width);
    return r;
}

template <class T>
__device__ __forceinline__ T wave_incl_scan(T v)
{
    const int lane = lane_id();
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const T t = shfl_up_any(v, o);
        if (lane >= o) v += t;
    }
    return v;
}

// Exclusive scan across a block of BS threads; *total receives the block sum.
// lds must hold BS/64 + 1 elements.  Contains __syncthreads: call from all
// threads of the block.
template <class T, int BS>
__device__ __forceinline__ T block_excl_scan(T v, T* lds, T* total)
{
    constexpr int NW = BS / kWave;
    const T inc = wave_incl_scan(v);
    const int w = threadIdx.x / kWave, lane = lane_id();
    if (lane == kWave - 1) lds[w] = inc;
    __syncthreads();
    if (w == 0) {
        const T s = lane < NW ? lds[lane] : T(0);
        const T si = wave_incl_scan(s);
        if (lane < NW) lds[lane] = si - s;
        if (lane == NW - 1) lds[NW] = si;
    }
    __syncthreads();
    const T res = inc - v + lds[w];
    *total = lds[NW];
    __syncthreads();
    return res;
}

// ---- Morton codes (x in the highest bit of each triple) --------------------
__device__ __forceinline__ uint32_t part1by2(uint32_t v)
{
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}
__device__ __forceinline__ uint32_t morton3(uint32_t x, uint32_t y, uint32_t z)
{
    return (part1by2(x) << 2) | (part1by2(y) << 1) | part1by2(z);
}

// Uniform grid description (device copy of the host's choice).
struct Grid {
    float lo[3];
    float inv_b;          // 1 / bin edge
    int dim[3];
    float h;              // the field's node spacing
    float org[3], inv_s;  // scaled coordinates of the index's boxes: (p - org) inv_s
    int root_lv;          // level of the field's tree root
};

__device__ __forceinline__ uint32_t grid_code(const Grid& g, float x, float y, float z)
{
    const float c[3] = {x, y, z};
    uint32_t b[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        float f = (c[k] - g.lo[k]) * g.inv_b;
        int i = (f >= 0.0f) ? (int)f : 0;           // NaN -> 0
        i = i < g.dim[k] ? i : g.dim[k] - 1;
        b[k] = (uint32_t)i;
    }
    return morton3(b[0], b[1], b[2]);
}

// Field of element x given the exclusive offsets off[0..nf] (off[0] = 0):
// the largest k < nf with off[k] <= x.
__device__ __forceinline__ int field_of(const int64_t* off, int nf, int64_t x)
{
    int lo = 0, hi = nf - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= x) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// Square root for lower bounds only: the hardware v_sqrt_f32 (within 1 ulp),
// not the correctly rounded sequence the build flags give sqrtf.  Every bound
// that uses it subtracts a relative slack of 2^-20 or more afterwards, which
// covers the 2^-23 relative error; a flushed tiny input gives 0, still a
// lower bound.
__device__ __forceinline__ float sqrt_lb(float x) { return __builtin_amdgcn_sqrtf(x); }

// ---- FP64 vector helpers (index build, FP64 settle) -------------------------
__device__ inline double dot3d(const double* u, const double* v)
{
    return u[0] * v[0] + u[1] * v[1] + u[2] * v[2];
}
__device__ inline void cross3d(const double* u, const double* v, double* w)
{
    w[0] = u[1] * v[2] - u[2] * v[1];
    w[1] = u[2] * v[0] - u[0] * v[2];
    w[2] = u[0] * v[1] - u[1] * v[0];
}

// ---- FP64 point-triangle distance (the search's final word) -----------------
// Squared distance from x to triangle abc (float points, arithmetic in
// FP64): the plane distance when the projection of x falls inside (edge
// functions n.(e x (x - v)) >= 0 for the three edges), else the nearest of
// the three edge segments; nearly collinear vertices (|n|^2 <= 1e-14 lmax^2)
// use the segments only.  Each difference (x - v, an edge) is formed from the
// float inputs where it is used, the same way each time, and each segment
// distance is taken beside its edge function, so few doubles are live at
// once: this runs at the end of the search kernel, whose occupancy depends on
// its register count.
__device__ inline void diff3d(const float* u, const float* v, double* w)
{
    for (int k = 0; k < 3; k++) w[k] = (double)u[k] - (double)v[k];
}

// Squared distance from the point at ax (relative to a) to the segment a,
// a + ab.
__device__ inline double seg_dist2_rel(const double* ax, const double* ab)
{
    const double l2 = dot3d(ab, ab);
    double t = l2 > 0.0 ? dot3d(ax, ab) / l2 : 0.0;
    t = fmin(fmax(t, 0.0), 1.0);
    double r = 0.0;
    for (int k = 0; k < 3; k++) { const double q = ax[k] - t * ab[k]; r += q * q; }
    return r;
}

__device__ inline double tri_dist2_f64(const float* x, const float* a, const float* b, const float* c)
{
    double n[3], nn, lmax;
    {
        double e0[3], e1[3], e2[3];
        diff3d(b, a, e0);
        diff3d(c, b, e1);
        diff3d(a, c, e2);
        cross3d(e0, e1, n);
        nn = dot3d(n, n);
        lmax = fmax(dot3d(e0, e0), fmax(dot3d(e1, e1), dot3d(e2, e2)));
    }
    bool inside = nn > 1e-14 * lmax * lmax;
    const float* v[3] = {a, b, c};
    const float* w[3] = {b, c, a};
    double hgt = 0.0, sd[3];
    for (int q = 0; q < 3; q++) {
        double xv[3], e[3], t[3];
        diff3d(x, v[q], xv);
        diff3d(w[q], v[q], e);
        if (q == 0) hgt = dot3d(n, xv);
        cross3d(e, xv, t);
        inside = inside && dot3d(n, t) >= 0.0;
        sd[q] = seg_dist2_rel(xv, e);
    }
    if (inside) return hgt * hgt / nn;
    return fmin(sd[0], fmin(sd[1], sd[2]));
}

// ---- FP32 point-triangle distance -------------------------------------------
// Triangle record (80 B): an orthonormal frame at vertex a, built in FP64
// when the index is built, with u along ab (the longest edge), the unit normal
// n and v = n x u; in it the triangle is (0,0), (B,0), (Cx,Cy), Cy >= 0:
//   a = (a, Cx - B)  u = (u, B)  v = (v, Cx)  n = (n, Cy)
//   i = (1/B, 1/|ac|^2, 1/|bc|^2, id)
// (inverse lengths are 0 for zero-length edges; id as bits, the top one set
// for collinear vertices, which have no interior and whose distance is that
// of the edge segments).  The point is projected once (X, Y, Z); the in-plane
// distance is 0 inside the triangle, else the nearest clamped edge
// projection; d^2 = d2D^2 + Z^2.  With ab the longest edge the 2D problem
// stays well conditioned however thin the triangle is, so no case needs FP64
// at query time.
struct TriRec {
    float4 a, u, v, n, i;
};
__device__ __forceinline__ int32_t tri_id(const TriRec& r) { return __float_as_int(r.i.w) & INT32_MAX; }

__device__ __forceinline__ float tri_dist2(float x, float y, float z, const TriRec& r)
{
    const float wx = x - r.a.x, wy = y - r.a.y, wz = z - r.a.z;
    const float X = __fmaf_rn(wz, r.u.z, __fmaf_rn(wy, r.u.y, wx * r.u.x));
    const float Y = __fmaf_rn(wz, r.v.z, __fmaf_rn(wy, r.v.y, wx * r.v.x));
    const float Z = __fmaf_rn(wz, r.n.z, __fmaf_rn(wy, r.n.y, wx * r.n.x));
    const float B = r.u.w, Cx = r.v.w, Cy = r.n.w, dCx = r.a.w;
    const float xb = X - B;
    const bool inside = (int)(Y >= 0.0f) & (int)(__fmaf_rn(Cy, X, -Cx * Y) >= 0.0f) &
                        (int)(__fmaf_rn(dCx, Y, -Cy * xb) >= 0.0f) & (int)(__float_as_int(r.i.w) >= 0);
    // edge ab
    float t = fminf(fmaxf(X * r.i.x, 0.0f), 1.0f);
    float ex = __fmaf_rn(-t, B, X);
    float d = __fmaf_rn(Y, Y, ex * ex);
    // edge ac
    t = fminf(fmaxf(__fmaf_rn(Y, Cy, X * Cx) * r.i.y, 0.0f), 1.0f);
    ex = __fmaf_rn(-t, Cx, X);
    float ey = __fmaf_rn(-t, Cy, Y);
    d = fminf(d, __fmaf_rn(ey, ey, ex * ex));
    // edge bc
    t = fminf(fmaxf(__fmaf_rn(Y, Cy, xb * dCx) * r.i.z, 0.0f), 1.0f);
    ex = __fmaf_rn(-t, dCx, xb);
    ey = __fmaf_rn(-t, Cy, Y);
    d = fminf(d, __fmaf_rn(ey, ey, ex * ex));
    return __fmaf_rn(Z, Z, inside ? 0.0f : d);
}

}  // namespace ftd
