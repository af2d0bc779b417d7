// cmg_learn.hip -- the learned tile smoother on gfx950: data gathering from a
// grid, FP32 training kernels (forward, loss, backward, weight gradients), the
// Adam update, and BF16 MFMA inference.
//
// Network (no reference counterpart): a 3-layer 3D conv net on one halo'd 10^3
// tile, 1 -> 16 -> 16 -> 1 channels, 3^3 kernels, zero "same" padding, ReLU
// after layers 1 and 2, no biases (so net(c x) = c net(x) for c > 0).  Weights
// are one flat array of 7776 floats: W1[16][27], W2[16 out][16 in][27],
// W3[16 in][27]; tap (di+1)*9 + (dj+1)*3 + (dk+1).  Volume index (i*10+j)*10+k.
// Input feature of a cell: r / D on INTERIOR cells of LEAF tiles of the tile's
// level (0 elsewhere); the output on the tile's own 8^3 cells is a correction
// of x.  Loss of a tile: sum over the interior 8^3 of (7-point Laplacian of
// (y - e))^2, mean over the batch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "cmg_device.hpp"
#include "cmg_kernels.hpp"

#pragma clang fp contract(off)

namespace cmg {
namespace k {

constexpr int NV = 1000, NC = 16, NW = 7776, OW2 = 432, OW3 = 7344;

__device__ __forceinline__ int vid(int i, int j, int k) { return (i * 10 + j) * 10 + k; }

// round to the nearest bfloat16 (ties to even) and back; NaN is kept quiet
__device__ __forceinline__ float bf16_round(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return f;
    u += 0x7fffu + ((u >> 16) & 1u);
    return __uint_as_float(u & 0xffff0000u);
}

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma32(s16x8 a, s16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// offset of tap t (0..26) in a volume of edge E
__device__ __forceinline__ int tap_off(int t, int E) { return (t / 9 - 1) * E * E + ((t / 3) % 3 - 1) * E + (t % 3 - 1); }

__device__ __forceinline__ uint16_t bf16_bits(float f) { return uint16_t(__float_as_uint(bf16_round(f)) >> 16); }

// (one instruction; NaN gives 0)
__device__ __forceinline__ float relu(float x) { return __builtin_amdgcn_fmed3f(x, 0.0f, INFINITY); }

__device__ __forceinline__ uint32_t pack_relu_bf16(float lo, float hi)
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{relu(lo), relu(hi)}, b16x2));
}

// ---------------------------------------------------------------- gather ----
// one halo'd 10^3 volume per tile of `list`: mode 0 the input feature r / D,
// mode 1 the raw value; cells of the tile and of its same-level LEAF
// neighbours (INTERIOR only), 0 elsewhere (corners of the volume included)
__global__ __launch_bounds__(256) void gather_tiles(TopoView tp, const int32_t* __restrict__ tiles, int n,
                                                    const float* __restrict__ V, const float* __restrict__ D, int mode,
                                                    float* __restrict__ out)
{
    const int b = blockIdx.x;
    if (b >= n) return;
    const int t = tiles[b];
    for (int p = threadIdx.x; p < NV; p += blockDim.x) {
        const int i = p / 100 - 1, j = (p / 10) % 10 - 1, kk = p % 10 - 1;
        const int out_axes = (i < 0 || i > 7) + (j < 0 || j > 7) + (kk < 0 || kk > 7);
        float val = 0.0f;
        if (out_axes <= 1) {
            int tt = t, l[3] = {i, j, kk};
            if (out_axes == 1) {
                const int a = (i < 0 || i > 7) ? 0 : (j < 0 || j > 7) ? 1 : 2;
                const bool neg = l[a] < 0;
                tt = tp.nbr[size_t(t) * 6 + (neg ? a : a + 3)];
                l[a] = neg ? 7 : 0;
                if (tt >= 0 && !(tp.ttype[tt] & LEAF)) tt = -1;
            }
            if (tt >= 0) {
                const size_t idx = size_t(tt) * 512 + cidx(l[0], l[1], l[2]);
                if (tp.ctype[idx] & INTERIOR) {
                    const float v = V[idx];
                    if (mode == 0) {
                        const float d = D[idx];
                        val = d != 0 ? v / d : 0.0f;
                    } else {
                        val = v;
                    }
                }
            }
        }
        out[size_t(b) * NV + p] = val;
    }
}

// ---------------------------------------------------------------- training ----
// One workgroup (512 threads, 8 wave64s) per chunk of tiles, everything of a tile in LDS.  BF16:
// weights and activations are rounded to bfloat16 in the forward pass (FP32 accumulation);
// the backward pass is FP32.
//
// Every convolution and weight gradient is a product on the matrix cores.  With 16 positions
// of the volume (or the 27 taps) along N and K in steps of four,
//   a1[co][p]     = sum over taps            W1[co][t] x[p + off t]             (K: 28 taps)
//   a2[co][p]     = sum over taps, ci        W2[co][ci][t] a1[ci][p + off t]    (BF16: K: 2 taps x 16 ci)
//   U[t][q]       = sum over ci              W3[ci][t] a2[ci][q],   y[p] = sum of U[t][p + off t]
//   dW3[ci][t]    = sum over q               a2[ci][q] g[q - off t]
//   g2[ci][q]     = sum over taps            W3[ci][t] g[q - off t]             (where a2 > 0)
//   dW2[co][ci]   = sum over p, tap by tap   g2[co][p] a1[ci][p + off t]
//   g1[ci][p]     = sum over taps, co        W2[co][ci][t] g2[co][p - off t]    (where a1 > 0)
//   dW1[co][t]    = sum over p               g1[co][p] x[p + off t]
// the FP32 ones on v_mfma_f32_16x16x4_f32, BF16's a2 on v_mfma_f32_16x16x32_bf16.  The two
// products with 6.9 M multiplications, dW2 and g1, bound it: 13,600 of a tile's 16,000 FP32
// MFMAs of 32 cycles, 53 us of a tile's time on the four SIMDs of a CU.  dW2's 27 taps are
// dealt to four pairs of waves, seven accumulators each, a pair's waves taking half the
// positions, so that one load of g2 serves seven products; g1 goes tap by tap over a wave's
// eight blocks of positions, so that four registers hold the weights in use.  Volumes read
// with an offset are zero-padded (x, g) or read through a mask of the taps that stay inside
// (vm); channel rows are 1,012 floats apart, which puts 16 rows, and 4 rows of 16 positions,
// on distinct banks.  (MI355X, 4,096 tiles, BF16: 2.03 ms, 127 us a tile, 92 TFLOP/s; 46.8 ms with
// one FMA a multiplication on the vector units, every operand from LDS and the weights from
// global memory.  Its gradients were 5e-8 from the 64-bit ones in FP32 mode, 8e-8 before.)
constexpr int TS = 1012;   // floats from one channel's 1,000 positions to the next's (the rest 0)
constexpr int NBLK = (NV + 15) / 16;   // 63 blocks of 16 positions

struct TrainLds {
    float xp[1728], gp[1728], sp[1728];   // 12^3, zero rim: x; y - e, then dL/dy; the interior Laplacian of y - e
    uint32_t vm[1008];                    // bit t: position + off t is inside the volume
    uint16_t pt[1008];                    // the position's place in the 12^3 volumes
    // FP32: a1 [16][TS]; BF16: a1 [2 halves of 8 channels][1000][8] and a2 [4 quarters of 4][1000][4],
    // bfloat16; then g1 [16][TS]
    float r0[16 * TS];
    float g2[16 * TS];                    // FP32: a2, then g2; BF16: U[9][1000], then g2
    float w1[7][64], w3[7][64];           // layers 1 and 3 as operands (row lane & 15, tap 4 s + lane / 16)
    float w3u[3][4][64];                  // layer 3 for U (row tap 9 g + lane & 15, channel 4 kk + lane / 16)
    double red[8];
};
static_assert(sizeof(TrainLds) <= 160 * 1024, "a CU's LDS");
constexpr int kA2 = 32000, kZero = 64000;   // bytes into r0 (BF16): a2, 16 zero bytes

// weights in the order the MFMA operands take them: [27 taps][4][64 lanes] for g1 (row ci = lane & 15,
// column co = 4 kk + lane / 16), then for a2 the same by (co, ci), or with BF16 [14 tap pairs][64 lanes][8]
constexpr int NPACK = 2 * 27 * 256;

template <bool BF16>
__global__ __launch_bounds__(256) void net_pack(const float* __restrict__ W, float* __restrict__ P)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e < 6912) {
        const int lane = e & 63, kk = (e >> 6) & 3, t = e >> 8;
        const int r = lane & 15, c = 4 * kk + (lane >> 4);
        const float b = W[OW2 + (c * NC + r) * 27 + t], f = W[OW2 + (r * NC + c) * 27 + t];
        P[e] = BF16 ? bf16_round(b) : b;
        if (!BF16) P[6912 + e] = f;
    }
    if (BF16 && e < 14 * 512) {
        const int j = e & 7, lane = (e >> 3) & 63, m = e >> 9;
        const int tap = 2 * m + (lane >> 5), ci = 8 * ((lane >> 4) & 1) + j;
        reinterpret_cast<uint16_t*>(P + 6912)[e] = tap < 27 ? bf16_bits(W[OW2 + ((lane & 15) * NC + ci) * 27 + tap]) : uint16_t(0);
    }
}

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ float bf16_float(uint16_t v) { return __uint_as_float(uint32_t(v) << 16); }

template <bool BF16>
__global__ __launch_bounds__(512) void net_train(const float* __restrict__ X, const float* __restrict__ E,
                                                 const int32_t* __restrict__ idx, int n, int per_wg,
                                                 const float* __restrict__ W, const float* __restrict__ Wp,
                                                 float* __restrict__ gpart, double* __restrict__ lpart)
{
    extern __shared__ __align__(16) unsigned char smem[];
    TrainLds& s = *reinterpret_cast<TrainLds*>(smem);
    unsigned char* const r0 = reinterpret_cast<unsigned char*>(s.r0);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, grp = lane >> 4;
    auto rnd = [](float v) { return BF16 ? bf16_round(v) : v; };
    for (int e = tid; e < 1728; e += 512) s.xp[e] = s.gp[e] = s.sp[e] = 0.0f;
    for (int e = tid; e < 16 * TS; e += 512) s.r0[e] = s.g2[e] = 0.0f;
    for (int p = tid; p < 1008; p += 512) {
        uint32_t m = 0;
        const int i = p / 100, j = (p / 10) % 10, kk = p % 10;
        for (int t = 0; t < 27; ++t) {
            const int a = i + t / 9 - 1, b = j + (t / 3) % 3 - 1, c = kk + t % 3 - 1;
            if (p < NV && unsigned(a) < 10u && unsigned(b) < 10u && unsigned(c) < 10u) m |= 1u << t;
        }
        s.vm[p] = m;
        s.pt[p] = uint16_t(p < NV ? ((i + 1) * 12 + j + 1) * 12 + kk + 1 : 0);
    }
    float *const w1f = &s.w1[0][0], *const w3f = &s.w3[0][0], *const w3uf = &s.w3u[0][0][0];
    for (int e = tid; e < 7 * 64; e += 512) {
        const int t = 4 * (e >> 6) + ((e >> 4) & 3), r = e & 15;
        w1f[e] = t < 27 ? rnd(W[r * 27 + t]) : 0.0f;
        w3f[e] = t < 27 ? rnd(W[OW3 + r * 27 + t]) : 0.0f;
    }
    for (int e = tid; e < 12 * 64; e += 512) {
        const int g = e >> 8, ci = 4 * ((e >> 6) & 3) + ((e >> 4) & 3), r = e & 15;
        w3uf[e] = r < 9 ? rnd(W[OW3 + ci * 27 + 9 * g + r]) : 0.0f;
    }
    int o12[7], oc[2];   // offsets of the operands' taps 4 s + grp, and of the weight gradients' column taps
#pragma unroll
    for (int e = 0; e < 7; ++e) o12[e] = 4 * e + grp < 27 ? tap_off(4 * e + grp, 12) : 0;
#pragma unroll
    for (int e = 0; e < 2; ++e) oc[e] = 16 * e + col < 27 ? tap_off(16 * e + col, 12) : 0;
    const int tap0 = 7 * (wave >> 1), half = wave & 1;   // the wave's share of dW2
    // gradients of the workgroup's tiles
    f32x4 G2[7], G3[2], G1[2];
#pragma unroll
    for (int m = 0; m < 7; ++m) G2[m] = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 2; ++e) G3[e] = G1[e] = f32x4{0, 0, 0, 0};
    double lacc = 0;
    __syncthreads();
    uint32_t vmb[8];   // the masks of the wave's blocks of positions
#pragma unroll
    for (int b = 0; b < 8; ++b) vmb[b] = s.vm[min(16 * (wave + 8 * b) + col, 1007)];
    auto block_pos = [&](int b) { return 16 * (wave + 8 * b) + col; };
    // g[16 out][p] = sum over taps and 16 in of P[t][in][out] src[in][p + (or -) off t] for the
    // wave's eight blocks; src channel rows of TS floats
    auto conv16 = [&](const float* __restrict__ Pw, const float* src, bool flip, f32x4 (&acc)[8]) {
#pragma unroll
        for (int b = 0; b < 8; ++b) acc[b] = f32x4{0, 0, 0, 0};
        float w[4];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) w[kk] = Pw[kk * 64 + lane];
#pragma unroll 1
        for (int t = 0; t < 27; ++t) {
            float wn[4] = {w[0], w[1], w[2], w[3]};
            if (t < 26) {
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) wn[kk] = Pw[((t + 1) * 4 + kk) * 64 + lane];
            }
            const int u = flip ? 26 - t : t, off = tap_off(u, 10);
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const float* q = src + grp * TS + ((vmb[b] >> u) & 1u ? block_pos(b) + off : NV);   // NV: zeros
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) acc[b] = mfma4(w[kk], q[kk * 4 * TS], acc[b]);
            }
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) w[kk] = wn[kk];
        }
    };
    const int b0 = blockIdx.x * per_wg, b1 = min(n, b0 + per_wg);
    for (int bi = b0; bi < b1; ++bi) {
        const size_t b = idx ? size_t(idx[bi]) : size_t(bi);
        float ev[2];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const int p = tid + 512 * m;
            ev[m] = p < NV ? E[b * NV + p] : 0.0f;
            if (p < NV) s.xp[s.pt[p]] = rnd(X[b * NV + p]);
        }
        if (BF16 && tid < 4) reinterpret_cast<uint32_t*>(r0 + kZero)[tid] = 0u;
        __syncthreads();
        // layer 1
#pragma unroll 2
        for (int bk = 0; bk < 8; ++bk) {
            const int p = block_pos(bk), c = s.pt[min(p, 1007)];
            f32x4 acc = {0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 7; ++e) acc = mfma4(s.w1[e][lane], s.xp[max(c + o12[e], 0)], acc);
            if (p < NV) {
                if constexpr (BF16) {
                    uint2 v;
                    v.x = pack_relu_bf16(acc[0], acc[1]);
                    v.y = pack_relu_bf16(acc[2], acc[3]);
                    *reinterpret_cast<uint2*>(r0 + (grp >> 1) * 16000 + p * 16 + (grp & 1) * 8) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) s.r0[(4 * grp + e) * TS + p] = acc[e] > 0 ? acc[e] : 0.0f;
                }
            }
        }
        __syncthreads();
        // layer 2
        {
            f32x4 acc[8];
            if constexpr (BF16) {
#pragma unroll
                for (int bk = 0; bk < 8; ++bk) acc[bk] = f32x4{0, 0, 0, 0};
                const uint4* wq = reinterpret_cast<const uint4*>(Wp + 6912) + lane;
                uint4 w = wq[0];
#pragma unroll 1
                for (int m = 0; m < 14; ++m) {
                    const uint4 wn = m < 13 ? wq[64 * (m + 1)] : w;
                    const int tap = 2 * m + (grp >> 1);   // (tap 27 has zero weights; its bit is never set)
                    const int off = tap_off(tap, 10) * 16 + (grp & 1) * 16000;
                    const uint32_t bit = 1u << tap;
#pragma unroll
                    for (int bk = 0; bk < 8; ++bk) {
                        const int addr = (vmb[bk] & bit) ? block_pos(bk) * 16 + off : kZero;
                        acc[bk] = mfma32(__builtin_bit_cast(s16x8, w), *reinterpret_cast<const s16x8*>(r0 + addr), acc[bk]);
                    }
                    w = wn;
                }
            } else {
                conv16(Wp + 6912, s.r0, false, acc);
            }
#pragma unroll
            for (int bk = 0; bk < 8; ++bk) {
                const int p = block_pos(bk);
                if (p >= NV) continue;
                if constexpr (BF16) {
                    uint2 v;
                    v.x = pack_relu_bf16(acc[bk][0], acc[bk][1]);
                    v.y = pack_relu_bf16(acc[bk][2], acc[bk][3]);
                    *reinterpret_cast<uint2*>(r0 + kA2 + grp * 8000 + p * 8) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) s.g2[(4 * grp + e) * TS + p] = acc[bk][e] > 0 ? acc[bk][e] : 0.0f;
                }
            }
        }
        __syncthreads();
        // a2 of channel c at position q
        auto a2_at = [&](int c, int q) -> float {
            if constexpr (BF16) return bf16_float(*reinterpret_cast<const uint16_t*>(r0 + kA2 + (c >> 2) * 8000 + q * 8 + (c & 3) * 2));
            else return s.g2[c * TS + q];
        };
        // layer 3 and d = y - e
        {
            float y[2] = {0.0f, 0.0f};
            if constexpr (BF16) {
#pragma unroll 1
                for (int g = 0; g < 3; ++g) {
#pragma unroll 2
                    for (int bk = 0; bk < 8; ++bk) {
                        const int q = block_pos(bk);
                        f32x4 acc = {0, 0, 0, 0};
#pragma unroll
                        for (int kk = 0; kk < 4; ++kk) acc = mfma4(s.w3u[g][kk][lane], q < NV ? a2_at(4 * kk + grp, q) : 0.0f, acc);
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (q < NV && 4 * grp + e < 9) s.g2[(4 * grp + e) * NV + q] = acc[e];
                    }
                    __syncthreads();
#pragma unroll
                    for (int m = 0; m < 2; ++m) {
                        const int p = tid + 512 * m;
                        const uint32_t ok = p < NV ? s.vm[p] >> (9 * g) : 0u;
#pragma unroll
                        for (int t = 0; t < 9; ++t)
                            if ((ok >> t) & 1u) y[m] += s.g2[t * NV + p + tap_off(9 * g + t, 10)];
                    }
                    __syncthreads();
                }
            } else {
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    const int p = tid + 512 * m;
                    for (int t = 0; t < 27; ++t) {
                        if (p >= NV || !((s.vm[p] >> t) & 1u)) continue;
                        for (int ci = 0; ci < NC; ++ci) y[m] = fmaf(W[OW3 + ci * 27 + t], s.g2[ci * TS + p + tap_off(t, 10)], y[m]);
                    }
                }
            }
#pragma unroll
            for (int m = 0; m < 2; ++m)
                if (tid + 512 * m < NV) s.gp[s.pt[tid + 512 * m]] = y[m] - ev[m];
        }
        __syncthreads();
        // s = interior Laplacian of d, loss
        double lt = 0;
        for (int p = tid; p < NV; p += 512) {
            const int i = p / 100, j = (p / 10) % 10, kk = p % 10, c = s.pt[p];
            float v = 0.0f;
            if (i >= 1 && i <= 8 && j >= 1 && j <= 8 && kk >= 1 && kk <= 8) {
                v = 6.0f * s.gp[c] - s.gp[c - 144] - s.gp[c + 144] - s.gp[c - 12] - s.gp[c + 12] - s.gp[c - 1] - s.gp[c + 1];
                lt += double(v) * double(v);
            }
            s.sp[c] = v;
        }
        lacc += lt;
        __syncthreads();
        // dL/dy = 2 Lap^T s / n
        const float sc = 2.0f / float(n);
        for (int p = tid; p < NV; p += 512) {
            const int c = s.pt[p];
            float v = 6.0f * s.sp[c];
            v -= s.sp[c - 144];
            v -= s.sp[c + 144];
            v -= s.sp[c - 12];
            v -= s.sp[c + 12];
            v -= s.sp[c - 1];
            v -= s.sp[c + 1];
            s.gp[c] = v * sc;
        }
        __syncthreads();
        // dL/dW3 (a2 before it is overwritten): the waves take every eighth group of four positions
        {
            f32x4 acc[2] = {f32x4{0, 0, 0, 0}, f32x4{0, 0, 0, 0}};
            for (int q0 = 4 * wave; q0 < NV; q0 += 32) {
                const int q = q0 + grp, c = s.pt[q];
                const float av = a2_at(col, q);
#pragma unroll
                for (int e = 0; e < 2; ++e) acc[e] = mfma4(av, s.gp[c - oc[e]], acc[e]);
            }
#pragma unroll
            for (int e = 0; e < 2; ++e) G3[e] += acc[e];
        }
        if (!BF16) __syncthreads();
        // dL/da2 masked by ReLU'
#pragma unroll 2
        for (int bk = 0; bk < 8; ++bk) {
            const int q = block_pos(bk), c = s.pt[min(q, 1007)];
            f32x4 acc = {0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 7; ++e) acc = mfma4(s.w3[e][lane], s.gp[max(c - o12[e], 0)], acc);
            if (q < NV) {
#pragma unroll
                for (int e = 0; e < 4; ++e) s.g2[(4 * grp + e) * TS + q] = a2_at(4 * grp + e, q) > 0 ? acc[e] : 0.0f;
            }
        }
        if (BF16 && tid < 16 * 12) s.g2[(tid / 12) * TS + NV + tid % 12] = 0.0f;   // (U was there)
        __syncthreads();
        // dL/dW2: the wave's seven taps over its half of the positions
        {
            f32x4 acc[7];
            int off[7];
#pragma unroll
            for (int m = 0; m < 7; ++m) {
                acc[m] = f32x4{0, 0, 0, 0};
                off[m] = tap_off(min(tap0 + m, 26), 10);
            }
            for (int p0 = 4 * half; p0 < NV; p0 += 8) {
                const int p = p0 + grp;
                const uint32_t ok = s.vm[p];
                const float av = s.g2[col * TS + p];
#pragma unroll
                for (int m = 0; m < 7; ++m) {
                    // 0 where the neighbour is outside (the load is inside LDS all the same)
                    const uint32_t in = uint32_t(-int((ok >> (tap0 + m)) & 1u));
                    uint32_t v;
                    if constexpr (BF16)
                        v = uint32_t(*reinterpret_cast<const uint16_t*>(r0 + (col >> 3) * 16000 + (p + off[m]) * 16 + (col & 7) * 2)) << 16;
                    else
                        v = __float_as_uint(*(reinterpret_cast<const float*>(r0) + col * TS + p + off[m]));
                    acc[m] = mfma4(av, __uint_as_float(v & in), acc[m]);
                }
            }
#pragma unroll
            for (int m = 0; m < 7; ++m) G2[m] += acc[m];
        }
        // dL/da1 masked by ReLU', in place of a1
        {
            f32x4 acc[8];
            conv16(Wp, s.g2, true, acc);
#pragma unroll
            for (int bk = 0; bk < 8; ++bk) {
                const int p = block_pos(bk);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    bool on = false;
                    if (p < NV) {
                        if constexpr (BF16)
                            on = bf16_float(*reinterpret_cast<const uint16_t*>(r0 + (grp >> 1) * 16000 + p * 16 + (grp & 1) * 8 + 2 * e)) > 0;
                        else
                            on = s.r0[(4 * grp + e) * TS + p] > 0;
                    }
                    acc[bk][e] = on ? acc[bk][e] : 0.0f;
                }
            }
            __syncthreads();
#pragma unroll
            for (int bk = 0; bk < 8; ++bk) {
                const int p = block_pos(bk);
                if (p >= NV) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e) s.r0[(4 * grp + e) * TS + p] = acc[bk][e];
            }
        }
        __syncthreads();
        // dL/dW1
        {
            f32x4 acc[2] = {f32x4{0, 0, 0, 0}, f32x4{0, 0, 0, 0}};
            for (int p0 = 4 * wave; p0 < NV; p0 += 32) {
                const int p = p0 + grp, c = s.pt[p];
                const float av = s.r0[col * TS + p];
#pragma unroll
                for (int e = 0; e < 2; ++e) acc[e] = mfma4(av, s.xp[c + oc[e]], acc[e]);
            }
#pragma unroll
            for (int e = 0; e < 2; ++e) G1[e] += acc[e];
        }
        __syncthreads();
    }
    // the workgroup's gradients: dW2 from the two halves, dW1 and dW3 from the eight waves
    float* out = gpart + size_t(blockIdx.x) * NW;
    if (half) {
#pragma unroll
        for (int m = 0; m < 7; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) s.r0[((wave >> 1) * 7 + m) * 256 + (4 * grp + e) * 16 + col] = G2[m][e];
    }
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int at = wave * 512 + (4 * grp + e) * 32 + 16 * k + col;
            s.g2[at] = G1[k][e];
            s.g2[4096 + at] = G3[k][e];
        }
    __syncthreads();
    if (!half) {
#pragma unroll
        for (int m = 0; m < 7; ++m) {
            const int t = tap0 + m;
            if (t >= 27) continue;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int co = 4 * grp + e;
                out[OW2 + (co * NC + col) * 27 + t] = G2[m][e] + s.r0[((wave >> 1) * 7 + m) * 256 + co * 16 + col];
            }
        }
    }
    for (int e = tid; e < 432; e += 512) {
        const int at = (e / 27) * 32 + e % 27;
        float v1 = 0.0f, v3 = 0.0f;
        for (int w = 0; w < 8; ++w) {
            v1 += s.g2[w * 512 + at];
            v3 += s.g2[4096 + w * 512 + at];
        }
        out[e] = v1;
        out[OW3 + e] = v3;
    }
    const double lb = block_sum(lacc, s.red);
    if (tid == 0) lpart[blockIdx.x] = lb;
}

// grad[w] = sum over workgroups of the partials (fixed order, FP64); loss likewise.  Few waves
// with a long sum each: 32 partials are in flight at a time (MI355X, 256 workgroups:
// 10 us, 72 us with one load in flight a thread)
__global__ __launch_bounds__(64) void net_reduce(const float* __restrict__ gpart, const double* __restrict__ lpart, int nwg,
                                                 int n, float* __restrict__ grad, double* __restrict__ loss)
{
    const int wi = blockIdx.x * blockDim.x + threadIdx.x;
    if (wi < NW) {
        double acc = 0;
        int g = 0;
        for (; g + 32 <= nwg; g += 32) {
            float v[32];
#pragma unroll
            for (int e = 0; e < 32; ++e) v[e] = gpart[size_t(g + e) * NW + wi];
#pragma unroll
            for (int e = 0; e < 32; ++e) acc += double(v[e]);
        }
        for (; g < nwg; ++g) acc += double(gpart[size_t(g) * NW + wi]);
        grad[wi] = float(acc);
    }
    if (blockIdx.x == gridDim.x - 1) {
        // the loss, its partials read a wave at a time
        double l = 0;
        for (int g0 = 0; g0 < nwg; g0 += 64) {
            const double v = g0 + int(threadIdx.x) < nwg ? lpart[g0 + threadIdx.x] : 0.0;
            for (int e = 0; e < 64; ++e) l += __shfl(v, e, 64);
        }
        if (threadIdx.x == 0) *loss = l / double(n);
    }
}

// Adam (Kingma and Ba, 2015), step t >= 1, FP32 state
__global__ __launch_bounds__(256) void adam(float* __restrict__ W, float* __restrict__ M, float* __restrict__ Vs,
                                            const float* __restrict__ G, int t, float lr, float b1, float b2, float eps)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= NW) return;
    const float c1 = 1.0f - powf(b1, float(t)), c2 = 1.0f - powf(b2, float(t));
    const float g = G[i];
    const float m = b1 * M[i] + (1.0f - b1) * g;
    const float v = b2 * Vs[i] + (1.0f - b2) * g * g;
    M[i] = m;
    Vs[i] = v;
    W[i] = W[i] - lr * (m / c1) / (sqrtf(v / c2) + eps);
}

// -------------------------------------------------------------- inference ----
// BF16 MFMA forward pass on the tile's own 8^3 cells: y = net(x), x gathered
// from channel R / D as for training.  Persistent: each 512-thread workgroup
// (8 wave64s) walks the tiles of a list.
// All three layers run on v_mfma_f32_16x16x32_bf16 with output channels as the M side and 16
// positions as the N side:
//   layer 1: [16 co x 32 (27 taps + 5 zero)] x [32 x 16 positions of the 10^3 volume]
//   layers 2 and 3: per pair of the nine taps in a plane, [16 rows x 32 (2 taps x 16 ci)] x [32 x
//            16 positions of one plane], 5 pairs (the tenth tap zero).  In layer 2 an operand of plane
//            i serves the outputs of planes i - 1, i and i + 1 with the weights of three taps across
//            the planes: 50 operands and 140 products for the ten planes of a column of positions.
//            Layer 3 has one output channel, so its rows are the three taps across the planes and
//            output i adds row 0 of plane i - 1, row 1 of plane i and row 2 of plane i + 1; it runs
//            on the tile's own 8^3 cells.
// Activations are rounded to bfloat16 after each ReLU, products accumulate in
// FP32 (the same rounding points as the training forward pass in BF16 mode).
// The input of the next tile (r / D on 512 own and 384 face-halo cells, 1.75
// cells per thread) is loaded into registers while the current tile's layer 3
// is computed; the neighbours come from the tile's 32-byte halo record.
// What bounds it is the issue of vector instructions (26.4 million a call on 3,680 tiles, 44 us of
// it), the LDS reads (27 million cycles of 256 CUs, 44 us) and the matrix cores (36 us), which
// overlap in part, and a last round of tiles that is not full.  Operands one tap pair at a time
// cost 1,330 reads of 1 KB a tile (630 now) and, without the zeros around a1, a test of the tap's
// place for each.  3,680 tiles of sphere-256: 217 -> 82 us (256 threads a workgroup, one block of
// positions after another: 217; tap pairs outermost, weights loaded once for 16 blocks: 174; 512
// threads, so four waves a SIMD: 141; zeros around a1: 113).
// LDS (81,648 B, two workgroups per CU).  Activations are stored by channel half so that the 16
// positions one MFMA operand reads are contiguous but for the holes (few bank conflicts):
//   [0, 44912)        a1, bf16 [2 halves of 8 ch][positions][8 ch].  Rows and planes of 10 are 11
//                     apart and 133 places lie before, between and after the halves: whatever a
//                     tap reads outside the volume is one of these zeros
//   [44912, 77232)    a2, bf16 [2 halves of 8 ch][10 planes][100 positions and a zero][8 ch]
//   [77232, 80688)    x on the zero-padded 12^3 volume, bf16 (edges and corners of the 10^3
//                     volume and the padding stay 0)
//   [80688, 81648)    layer 3's weights, bf16 [5 pairs][2 taps][2 halves of 8 ci][3 planes][8 ci]
constexpr int IL_A1 = 0, IL_A2 = 44912, IL_X = 77232, IL_W3 = 80688, IL_BYTES = 81648;
static_assert(2 * IL_BYTES <= 160 * 1024, "two workgroups' LDS on a CU");
constexpr int IL_HALF = 1343 * 16;   // from a1's lower channels to its upper ones
__device__ __forceinline__ int a1_place(int i, int j, int k) { return IL_A1 + (133 + (i * 11 + j) * 11 + k) * 16; }
constexpr int IN_PT = 2;   // input cells per thread (896 = 512 own + 384 halo, 512 threads)

// registers of one tile's input: padded-volume position (-1: none), r, D, cell type
struct InferIn {
    int pos[IN_PT];
    float r[IN_PT], d[IN_PT];
    uint8_t ct[IN_PT];
};

__device__ __forceinline__ void infer_issue(InferIn& in, const TopoView& tp, int t, const float* __restrict__ R,
                                            const float* __restrict__ D)
{
#pragma unroll
    for (int m = 0; m < IN_PT; ++m) {
        in.pos[m] = -1;
        in.r[m] = 0.0f;
        in.d[m] = 0.0f;
        in.ct[m] = 0;
    }
    if (t < 0) return;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // (places kept over the tiles would spill)
    const int4* hr = reinterpret_cast<const int4*>(tp.halo + size_t(t) * 8);
    const int4 ha = hr[0], hb = hr[1];
    const int nb[6] = {ha.x, ha.y, ha.z, ha.w, hb.x, hb.y};
    const uint32_t ty03 = uint32_t(hb.z), ty45 = uint32_t(hb.w);
#pragma unroll
    for (int m = 0; m < IN_PT; ++m) {
        const int e = tid + 512 * m;
        if (e >= 896) continue;
        int tt, l0, l1, l2, p0, p1, p2;   // source tile, its cell, padded position
        if (e < 512) {
            tt = t;
            l0 = e >> 6; l1 = (e >> 3) & 7; l2 = e & 7;
            p0 = l0 + 2; p1 = l1 + 2; p2 = l2 + 2;
        } else {
            const int k = e - 512, f = k >> 6, fi = k & 63, axis = f >> 1;
            const bool neg = !(f & 1);
            const int slot = neg ? axis : axis + 3;
            int nt = nb[0];
            nt = slot == 1 ? nb[1] : nt;
            nt = slot == 2 ? nb[2] : nt;
            nt = slot == 3 ? nb[3] : nt;
            nt = slot == 4 ? nb[4] : nt;
            nt = slot == 5 ? nb[5] : nt;
            const uint32_t nty = (slot < 4 ? ty03 >> (8 * slot) : ty45 >> (8 * (slot - 4))) & 0xffu;
            tt = (nt >= 0 && (nty & LEAF)) ? nt : -1;
            const int a = fi >> 3, bq = fi & 7, lo = neg ? 7 : 0, po = neg ? 1 : 10;
            if (axis == 0) { l0 = lo; l1 = a; l2 = bq; p0 = po; p1 = a + 2; p2 = bq + 2; }
            else if (axis == 1) { l0 = a; l1 = lo; l2 = bq; p0 = a + 2; p1 = po; p2 = bq + 2; }
            else { l0 = a; l1 = bq; l2 = lo; p0 = a + 2; p1 = bq + 2; p2 = po; }
        }
        in.pos[m] = (p0 * 12 + p1) * 12 + p2;
        if (tt >= 0) {
            const size_t idx = size_t(tt) * 512 + cidx(l0, l1, l2);
            in.ct[m] = tp.ctype[idx];
            in.d[m] = D[idx];
            in.r[m] = R[idx];
        }
    }
}

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void net_infer(TopoView tp, const int32_t* __restrict__ tiles, int n,
                                                 const float* __restrict__ R, const float* __restrict__ D,
                                                 const float* __restrict__ W, float* __restrict__ Y,
                                                 const double* __restrict__ S)
{
    extern __shared__ __align__(16) unsigned char lds[];
    if (stopped(S)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 15, grp = lane >> 4;
    // weights as MFMA A operands (row = col): layer 1 W1[co][tap 8 grp + j]
    s16x8 w1v;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int tap = 8 * grp + j;
        w1v[j] = tap < 27 ? short(bf16_bits(W[col * 27 + tap])) : short(0);
    }
    // layer-1 tap offsets on the padded 12^3 volume (taps 27..31 are zero taps)
    int o1[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) o1[j] = 8 * grp + j < 27 ? tap_off(8 * grp + j, 12) : 0;
    for (int e = tid; e < IL_X / 16; e += 512) reinterpret_cast<uint4*>(lds)[e] = make_uint4(0u, 0u, 0u, 0u);
    for (int e = tid; e < 1728 / 2; e += 512) reinterpret_cast<uint32_t*>(lds + IL_X)[e] = 0u;
    if (tid < 480) {
        const int j = tid & 7, d = (tid >> 3) % 3, g = (tid / 24) & 3, r = 2 * (tid / 96) + (g >> 1);
        reinterpret_cast<uint16_t*>(lds + IL_W3)[tid] = r < 9 ? bf16_bits(W[OW3 + (8 * (g & 1) + j) * 27 + 9 * d + r]) : uint16_t(0);
    }
    const uint16_t* xs = reinterpret_cast<const uint16_t*>(lds + IL_X);
    // per block of 16 positions of this wave (block wave + 8 b; the last ones lie beyond the volume:
    // computed like its last position and dropped) the places in x and in a1
    int place[8];   // of 2 bytes in x + 2048 times that of 16 in a1
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const int p = min(16 * (wave + 8 * b) + col, NV - 1), i = p / 100, j = (p / 10) % 10, kk = p % 10;
        place[b] = ((i + 1) * 12 + j + 1) * 12 + kk + 1 + a1_place(i, j, kk) / 16 * 2048;
    }
    // of layer 2's positions 16 wave + col of a plane, in the first plane
    const int p2 = min(16 * wave + col, 99), plane2 = a1_place(0, p2 / 10, p2 % 10);

    InferIn cur;
    infer_issue(cur, tp, blockIdx.x < n ? tiles[blockIdx.x] : -1, R, D);
    __syncthreads();
    for (int b = blockIdx.x; b < n; b += gridDim.x) {
        const int t = tiles[b];
        // input on the zero-padded 12^3 volume: r / D on INTERIOR cells of the
        // tile and of its same-level LEAF face neighbours, 0 elsewhere
#pragma unroll
        for (int m = 0; m < IN_PT; ++m)
            if (cur.pos[m] >= 0) {
                const float val = (cur.ct[m] & INTERIOR) && cur.d[m] != 0 ? cur.r[m] / cur.d[m] : 0.0f;
                reinterpret_cast<uint16_t*>(lds + IL_X)[cur.pos[m]] = bf16_bits(val);
            }
        __syncthreads();
        const int bn = b + int(gridDim.x);
        if (t < 0) {
            infer_issue(cur, tp, bn < n ? tiles[bn] : -1, R, D);
            continue;
        }
        // (an address for every block and operand, kept over the tiles, would spill)
#pragma unroll
        for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(o1[j]));
        int grp = lane >> 4;
        asm volatile("" : "+v"(grp));
        // layer 1 (taps 24, 25, 26 and zeros for the last lanes)
        const uint32_t m1[4] = {~0u, grp == 3 ? 0xffffu : ~0u, grp == 3 ? 0u : ~0u, grp == 3 ? 0u : ~0u};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int p = 16 * (wave + 8 * q) + col;
            const bool ok = p < NV;
            const int c12 = place[q] & 2047, c11 = (place[q] >> 11) * 16;
            uint32_t xw[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) xw[j] = (uint32_t(xs[c12 + o1[2 * j]]) | uint32_t(xs[c12 + o1[2 * j + 1]]) << 16) & m1[j];
            const s16x8 xv = __builtin_bit_cast(s16x8, make_uint4(xw[0], xw[1], xw[2], xw[3]));
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            acc = mfma32(w1v, xv, acc);
            if (ok) {
                uint2 v;
                v.x = pack_relu_bf16(acc[0], acc[1]);
                v.y = pack_relu_bf16(acc[2], acc[3]);
                *reinterpret_cast<uint2*>(lds + c11 + (grp >> 1) * IL_HALF + (grp & 1) * 8) = v;
            }
        }
        __syncthreads();
        // layer 2: wave w has positions 16 w .. of all ten planes
        if (wave < 7) {
            f32x4 acc[10];
#pragma unroll
            for (int i = 0; i < 10; ++i) acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            const uint4* wq = reinterpret_cast<const uint4*>(W + NW) + lane;   // (infer_pack)
            uint4 w[3] = {wq[0], wq[64], wq[128]};
#pragma unroll 1
            for (int m = 0; m < 5; ++m) {
                uint4 wn[3];
#pragma unroll
                for (int d = 0; d < 3; ++d) wn[d] = wq[64 * (3 * min(m + 1, 4) + d)];
                const int r = 2 * m + (grp >> 1);   // (no tap 9: the hole at the end of a row)
                const int at = (grp & 1) * IL_HALF + (r < 9 ? plane2 + ((r / 3 - 1) * 11 + r % 3 - 1) * 16 : a1_place(0, 0, 10));
#pragma unroll
                for (int i = 0; i < 10; ++i) {
                    const s16x8 x = *reinterpret_cast<const s16x8*>(lds + at + 1936 * i);
                    if (i > 0) acc[i - 1] = mfma32(__builtin_bit_cast(s16x8, w[2]), x, acc[i - 1]);
                    acc[i] = mfma32(__builtin_bit_cast(s16x8, w[1]), x, acc[i]);
                    if (i < 9) acc[i + 1] = mfma32(__builtin_bit_cast(s16x8, w[0]), x, acc[i + 1]);
                }
#pragma unroll
                for (int d = 0; d < 3; ++d) w[d] = wn[d];
            }
            const int p = 16 * wave + col;
            if (p < 100) {
#pragma unroll
                for (int i = 0; i < 10; ++i) {
                    uint2 v;
                    v.x = pack_relu_bf16(acc[i][0], acc[i][1]);
                    v.y = pack_relu_bf16(acc[i][2], acc[i][3]);
                    *reinterpret_cast<uint2*>(lds + IL_A2 + (grp >> 1) * 16160 + (grp & 1) * 8 + p * 16 + 1616 * i) = v;
                }
            }
        }
        __syncthreads();
        // the next tile's input loads fly while layer 3 runs (issued here, after
        // layer 2, whose register needs are the kernel's peak)
        infer_issue(cur, tp, bn < n ? tiles[bn] : -1, R, D);
        // layer 3 on the tile's cells: wave w has cells 16 (w & 3) .. of planes 4 (w >> 2) ..
        {
            f32x4 acc[6];
#pragma unroll
            for (int i = 0; i < 6; ++i) acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            const int c = wave & 3, h = wave >> 2;
            // rows 0..2 hold the weights of the three planes
            const unsigned char* w3 = lds + (col < 3 ? IL_W3 + (3 * grp + col) * 16 : IL_A1);
            const int ws = col < 3 ? 192 : 0;
            const int half = IL_A2 + (grp & 1) * 16160 + h * 6464;
#pragma unroll 1
            for (int m = 0; m < 5; ++m) {
                const int r = 2 * m + (grp >> 1);   // (no tap 9: the hole at the end of a plane)
                const int at = half + (r < 9 ? (2 * c + (col >> 3) + r / 3) * 160 + ((col & 7) + r % 3) * 16 : 1600);
                const s16x8 w = *reinterpret_cast<const s16x8*>(w3 + ws * m);
#pragma unroll
                for (int i = 0; i < 6; ++i) acc[i] = mfma32(w, *reinterpret_cast<const s16x8*>(lds + at + 1616 * i), acc[i]);
            }
            if (grp == 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const size_t cell = size_t(t) * 512 + 64 * (4 * h + q) + 16 * c + col;
                    Y[cell] = (tp.ctype[cell] & INTERIOR) ? acc[q][0] + acc[q + 1][1] + acc[q + 2][2] : 0.0f;
                }
            }
        }
    }
}

// the weights of layer 2 for net_infer, bf16: [5 pairs of in-plane taps][3 planes][64 lanes][8],
// row lane & 15 = output channel, in-plane tap 2 m + lane / 32, input channel 8 (lane / 16 & 1) + j
constexpr int IPACK = 15 * 512;
__global__ __launch_bounds__(256) void infer_pack(const float* __restrict__ W, uint16_t* __restrict__ P)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= IPACK) return;
    const int j = e & 7, lane = (e >> 3) & 63, d = (e >> 9) % 3, m = (e >> 9) / 3;
    const int r = 2 * m + (lane >> 5), ci = 8 * ((lane >> 4) & 1) + j;
    P[e] = r < 9 ? bf16_bits(W[OW2 + ((lane & 15) * NC + ci) * 27 + 9 * d + r]) : uint16_t(0);
}

// in-bounds check of the MFMA operand layouts: one wave64, C = A B for a
// 16 x K bf16 A and a K x 16 bf16 B (row-major bit patterns), K = 16 or 32
__global__ __launch_bounds__(64) void mfma_probe(int K, const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                                 float* __restrict__ C)
{
    const int lane = threadIdx.x, row = lane & 15, grp = lane >> 4;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    if (K == 32) {
        s16x8 av, bv;
        for (int e = 0; e < 8; ++e) {
            av[e] = short(A[row * 32 + 8 * grp + e]);
            bv[e] = short(B[(8 * grp + e) * 16 + row]);
        }
        acc = mfma32(av, bv, acc);
    } else {
        bf16x4 av, bv;
        for (int e = 0; e < 4; ++e) {
            av[e] = short(A[row * 16 + 4 * grp + e]);
            bv[e] = short(B[(4 * grp + e) * 16 + row]);
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, bv, acc, 0, 0, 0);
    }
    for (int e = 0; e < 4; ++e) C[(4 * grp + e) * 16 + row] = acc[e];
}
}  // namespace k

// ---------------------------------------------------------------- launchers ---

void launch_gather_tiles(const DevGrid& d, const int32_t* tiles, int n, const float* V, const float* D, int mode, float* out,
                         hipStream_t st)
{
    if (n <= 0) return;
    k::gather_tiles<<<n, 256, 0, st>>>(view(d), tiles, n, V, D, mode, out);
}

int launch_net_train(const float* X, const float* E, const int32_t* idx, int n, const float* W, float* wpack, float* gpart,
                     double* lpart, int max_wg, bool bf16, hipStream_t st)
{
    if (n <= 0) return 0;
    const int nwg = std::max(1, std::min(max_wg, n));
    const int per = (n + nwg - 1) / nwg;
    const int used = (n + per - 1) / per;
    const size_t lds = sizeof(k::TrainLds);
    static bool attr = [] {
        (void)hipFuncSetAttribute((const void*)k::net_train<true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  int(sizeof(k::TrainLds)));
        (void)hipFuncSetAttribute((const void*)k::net_train<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  int(sizeof(k::TrainLds)));
        return true;
    }();
    (void)attr;
    if (bf16) {
        k::net_pack<true><<<28, 256, 0, st>>>(W, wpack);
        k::net_train<true><<<used, 512, lds, st>>>(X, E, idx, n, per, W, wpack, gpart, lpart);
    } else {
        k::net_pack<false><<<28, 256, 0, st>>>(W, wpack);
        k::net_train<false><<<used, 512, lds, st>>>(X, E, idx, n, per, W, wpack, gpart, lpart);
    }
    return used;
}

size_t net_pack_floats() { return size_t(k::NPACK); }

size_t infer_pack_floats() { return size_t(k::IPACK / 2); }

void launch_infer_pack(const float* W, float* P, hipStream_t st)
{
    k::infer_pack<<<(k::IPACK + 255) / 256, 256, 0, st>>>(W, reinterpret_cast<uint16_t*>(P));
}

void launch_net_reduce(const float* gpart, const double* lpart, int nwg, int n, float* grad, double* loss, hipStream_t st)
{
    k::net_reduce<<<(k::NW + 63) / 64, 64, 0, st>>>(gpart, lpart, nwg, n, grad, loss);
}

void launch_adam(float* W, float* M, float* V, const float* G, int t, float lr, float b1, float b2, float eps, hipStream_t st)
{
    k::adam<<<(k::NW + 255) / 256, 256, 0, st>>>(W, M, V, G, t, lr, b1, b2, eps);
}

void launch_net_infer(const DevGrid& d, const LaunchList& l, const float* R, const float* D, const float* W, float* Y,
                      const double* S, hipStream_t st)
{
    if (l.n <= 0) return;
    static bool attr = [] {
        (void)hipFuncSetAttribute((const void*)k::net_infer, hipFuncAttributeMaxDynamicSharedMemorySize, k::IL_BYTES);
        return true;
    }();
    (void)attr;
    // persistent: two workgroups per CU
    const int grid = std::max(1, std::min(l.n, d.wg_cap / 4));
    k::net_infer<<<grid, 512, k::IL_BYTES, st>>>(view(d), l.d, l.n, R, D, W, Y, S);
}

void launch_mfma_probe(int K, const uint16_t* A, const uint16_t* B, float* C, hipStream_t st)
{
    k::mfma_probe<<<1, 64, 0, st>>>(K, A, B, C);
}

}  // namespace cmg
