// cmg_device.hpp -- device helpers shared by the kernel files.
#pragma once

#include <hip/hip_runtime.h>

#include "cmg_kernels.hpp"

#pragma clang fp contract(off)

namespace cmg {
namespace k {

// LDS index of a cell of the 10^3 halo'd tile (local coords -1..8)
__device__ __forceinline__ int SX(int i, int j, int k) { return (i + 1) * 100 + (j + 1) * 10 + (k + 1); }
__device__ __forceinline__ int cidx(int i, int j, int k) { return (i << 6) | (j << 3) | k; }

__device__ __forceinline__ bool stopped(const double* S) { return S && S[S_DONE] != 0.0; }

// the list entry of this workgroup, or -2 when the solve has stopped; the entry's
// load is issued before the stop test so that the two round trips overlap
__device__ __forceinline__ int list_tile(const int32_t* list, const double* S)
{
    const int t = list[blockIdx.x];
    return stopped(S) ? -2 : t;
}

// the entries of a coded level's table (the last one holds the tile spacing)
template <int Q>
constexpr int code_table() { return Q == 4 ? kWideCodes : kCodes; }

// a cell word's code of the face coefficient on axis a: bits 8a+8.. (forms 2, 3) or 10a+2.. (form 4)
template <int Q>
__device__ __forceinline__ uint32_t word_code(uint32_t w, int a)
{
    if constexpr (Q == 4) return (w >> (10 * a + 2)) & 0x3ffu;
    else return (w >> (8 * a + 8)) & 0xffu;
}

// a cell word's cell type: byte 0 (forms 2, 3), or 0..3 in bits 0-1 for 0, DIRICHLET, INTERIOR, NEUMANN (form 4)
template <int Q>
__device__ __forceinline__ uint8_t word_type(uint32_t w)
{
    if constexpr (Q == 4) return uint8_t((0x4210u >> (4 * (w & 3u))) & 0xfu);
    else return uint8_t(w);
}

template <int N, typename E>
struct alignas(N * sizeof(E)) Pack {
    E v[N];
};

// N consecutive elements at p (aligned to N elements) in one access
template <int N, typename E>
__device__ __forceinline__ void vload(const E* __restrict__ p, E (&out)[N])
{
    const Pack<N, E> pk = *reinterpret_cast<const Pack<N, E>*>(p);
#pragma unroll
    for (int i = 0; i < N; ++i) out[i] = pk.v[i];
}

template <int N, typename E>
__device__ __forceinline__ void vstore(E* __restrict__ p, const E (&in)[N])
{
    Pack<N, E> pk;
#pragma unroll
    for (int i = 0; i < N; ++i) pk.v[i] = in[i];
    *reinterpret_cast<Pack<N, E>*>(p) = pk;
}

// n / d for the FP64 reciprocal rd = 1 / d: the correctly rounded FP32 quotient.  The product
// is within 2^-50 of n / d, and no quotient of two FP32 numbers lies within 2^-49 of the
// midpoint of two neighbouring normal FP32 numbers.  A subnormal quotient can be a midpoint (d
// is then a multiple of 2), and the product just beside it: 6 % of such ties round to the other
// neighbour, 2^-149 off.  (A test for it, in the passes, takes 1 to 14 % of a uniform 64^3 solve.)
__device__ __forceinline__ float quotient(float n, double rd) { return float(double(n) * rd); }

// 1 / d to within 2^-51 (v_rcp_f64 and two Newton steps); +-inf for 0, 0 for +-inf, NaN for NaN
__device__ __forceinline__ double reciprocal(float d)
{
    const double v = d, r0 = __builtin_amdgcn_rcp(v);
    const double r1 = fma(fma(-v, r0, 1.0), r0, r0);
    const double r2 = fma(fma(-v, r1, 1.0), r1, r1);
    return r2 == r2 ? r2 : r0;
}

// one cell of a block kept in LDS: A x at LDS index c (strides si, sj, 1) with the face
// coefficients in registers (neg_lap's order)
__device__ __forceinline__ float block_lap(const float* x, int c, int si, int sj, float x0, const float (&cm)[3],
                                           const float (&cp)[3], float d)
{
    const float v0 = x[c - si], v1 = x[c + si], v2 = x[c - sj], v3 = x[c + sj], v4 = x[c - 1], v5 = x[c + 1];
    float r = x0 * d;
    r = fmaf(cm[0], v0, r);
    r = fmaf(cp[0], v1, r);
    r = fmaf(cm[1], v2, r);
    r = fmaf(cp[1], v3, r);
    r = fmaf(cm[2], v4, r);
    r = fmaf(cp[2], v5, r);
    return d == 0 ? 0.0f : r;
}

// consecutive cells, pairs swapped when odd: [2s] is then the pair's red cell, [2s + 1] its black one
template <int N, typename E>
__device__ __forceinline__ void by_colour(E (&v)[N], bool odd)
{
#pragma unroll
    for (int s = 0; s < N; s += 2) {
        const E a = v[s], b = v[s + 1];
        v[s] = odd ? b : a;
        v[s + 1] = odd ? a : b;
    }
}

// element s (0..5, thread-varying) of (a.x, a.y, a.z, a.w, b.x, b.y) by selects,
// with no private array (which the compiler would place in LDS)
__device__ __forceinline__ int pick6(int4 a, int4 b, int s)
{
    int r = a.x;
    r = s == 1 ? a.y : r;
    r = s == 2 ? a.z : r;
    r = s == 3 ? a.w : r;
    r = s == 4 ? b.x : r;
    r = s == 5 ? b.y : r;
    return r;
}

// element s (0..7, thread-varying) of (a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w) by selects
__device__ __forceinline__ int pick8(int4 a, int4 b, int s)
{
    int r = pick6(a, b, s);
    r = s == 6 ? b.z : r;
    r = s == 7 ? b.w : r;
    return r;
}

// A one-tile stencil workgroup's record (launch-list order, 7 x 16 bytes, read with
// scalar loads right after the launch): the tile, its level, type | octant << 8 and
// parent; its halo record (face neighbours, their tile types packed in bytes, own
// type in byte 7.3); the parents of the face neighbours and their octants (the
// operator's fresh GHOST values, the cycle's pulled prolongation); its children by
// octant (for a sweep that prolongs into them).  One round trip gives the workgroup every address it needs:
// the tile's own loads and its halo loads follow at once.
struct TileRec {
    int t, level, meta, parent;
    int4 ha, hb, ga, gb;
    int4 ca, cb;   // children by octant (CHILD records only)
    int tid;       // the thread's index among the threads working on the tile
};

// t = -1: padding entry, -2: the solve has stopped.  S is never null here (launches
// outside a solve pass the grid's idle block, whose flag is never set), so the stop
// flag is read with no branch and its load overlaps the record's.
template <bool FRESH, bool STOP = true, bool CHILD = false>
__device__ __forceinline__ TileRec rec_tile(const int4* __restrict__ rec, const double* __restrict__ S)
{
    const int4* r = rec + kRecWords * size_t(blockIdx.x);
    const int4 r0 = r[0];
    TileRec x;
    x.ha = r[1];
    x.hb = r[2];
    if (FRESH) {
        x.ga = r[3];
        x.gb = r[4];
    } else {
        x.ga = make_int4(-1, -1, -1, -1);
        x.gb = make_int4(-1, -1, 0, 0);
    }
    if (CHILD) {
        x.ca = r[5];
        x.cb = r[6];
    } else {
        x.ca = x.cb = make_int4(-1, -1, -1, -1);
    }
    x.t = (STOP && S[S_DONE] != 0.0) ? -2 : r0.x;
    x.tid = threadIdx.x;
    x.level = r0.y;
    x.meta = r0.z;
    x.parent = r0.w;
    return x;
}

__device__ __forceinline__ float rec_h(const TopoView& tp, const TileRec& r) { return tp.h0 / float(1 << r.level); }

// wave64 + workgroup reduction of one double per thread; result valid in thread 0
__device__ __forceinline__ double block_sum(double v, double* red)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) red[w] = v;
    __syncthreads();
    double s = 0;
    if (threadIdx.x == 0)
        for (int i = 0; i < int(blockDim.x >> 6); ++i) s += red[i];
    return s;
}

__device__ __forceinline__ float tile_h(const TopoView& tp, int t) { return tp.h0 / float(1 << tp.tlevel[t]); }

// Grid-stride loops over the tiles of a list, 128 threads x float4 per tile,
// two tiles per 256-thread workgroup step.  Launch lists hold Morton-consecutive
// tiles 8 entries apart (entry b is meant for a one-tile workgroup on XCD b % 8),
// so step w takes entries 16 (w / 8) + w % 8 and the one 8 after it: two Morton
// neighbours of the XCD that a workgroup w runs on.
#define CMG_TILE_LOOP(list, n)                                                                      \
    for (int w_ = blockIdx.x; 16 * (w_ >> 3) < (n); w_ += gridDim.x)                               \
        if (const int pos = 16 * (w_ >> 3) + (w_ & 7) + 8 * int(threadIdx.x >> 7); pos < (n))       \
            if (const int t_ = (list)[pos]; t_ >= 0)

__device__ __forceinline__ size_t quad_index(int t) { return size_t(t) * 128 + (threadIdx.x & 127); }

}  // namespace k
}  // namespace cmg
