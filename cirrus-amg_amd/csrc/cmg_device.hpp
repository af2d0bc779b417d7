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
// midpoint of two neighbouring normal FP32 numbers.
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
