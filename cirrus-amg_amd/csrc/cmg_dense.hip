// cmg_dense.hip -- a FAS cycle's visit to a complete level, in two launches.
//
// A level of 8^l tiles under a single root fills the domain: it has no GHOST tile, every
// neighbour cell is a cell of the level, and a smoothing pass depends on the 7-point
// neighbourhood alone.  So one workgroup can do all of a tile's passes without waiting for
// its neighbours' workgroups: it takes the tile with a halo as deep as the passes and
// computes the halo's cells again.
//   dense_visit<..., false>: the FAS save, the pre-smoothing, the residual and its
//     restriction (fas_save, gs_color or jacobi, residual_restrict); x goes from X to T and
//     the saved right-hand side to BN, since the neighbours still read X and B
//   dense_visit<..., true>: the prolongation from the level below, the post-smoothing, the
//     r.z partials and the prolongation to the level above (fas_prolong_v, gs_color or
//     jacobi); x goes from T to X, the saved right-hand side to B
// Every value is computed with the operations of the kernels named, so the results are the
// same bits, but where a quotient lies halfway between two subnormal numbers (quotient()).
//
// What bounds the kernels they replace on such levels is the latency of a launch, 4 to 5 us
// whatever its work: a red-black visit of two sweeps each way took eleven launches, a Jacobi
// visit five.  Here a workgroup of 512 threads holds the 16^3 cells within four of the tile,
// eight a thread, their coefficients in registers, x in LDS; cells too deep for a pass are
// mostly left out of it.  What bounds it is instruction issue (about 900 VALU instructions a
// wave, two waves a SIMD) and the loads of the halo, so a thread's cells are two rows of four
// (seven of the twelve neighbours of a colour's four cells are its own registers), a wave's
// rows have one parity, and a division is a product with an FP64 reciprocal.
// MI355X, W-cycle settings: a visit to 64 tiles 7.4 + 6.5 us, to 512 tiles 10.4 + 9.3 us,
// against 11 launches of 4.0 to 4.8 us.  At 4,096 tiles the halo's work is no longer hidden:
// the uniform 128^3 solve takes 3.54 ms this way and 2.77 ms with one launch a pass (V-cycle;
// W-cycle 3.10 and 3.05 ms), so levels of at most kDenseTiles = 512 tiles take it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdexcept>

#include "cmg_device.hpp"
#include "cmg_kernels.hpp"

#pragma clang fp contract(off)

namespace cmg {
namespace k {

struct DenseArgs {
    const int32_t* tab;   // kDenseWords per list entry: the 27 tiles around it, their parents, types
    const int4* rec;      // the level's tile records (level, children)
    float *X, *T, *B, *BN, *X0;
    Coef C;
    float Rr, P, w;
    double omega;
    int level, iters;
    int zero;    // pre: x is 0 (not read)
    int save;    // pre: the FAS save is due; post: it was done (the right-hand side is in BN)
    int push;    // post: prolong into the level above
    double* rz;  // post: r.z partials, one a list entry, or null
};

// x in LDS: 18 x 18 rows along k (the tile and five cells around it; of the outermost, the
// faces), at a row stride whose multiples spread a wave's 8 x 4 quads over the banks
constexpr int kRow = 21, kPlane = 18 * kRow;

template <int Q>
struct DenseLds {
    float x[18 * kPlane];
    float v[512];            // pre: residuals; post: x of the tile
    float v0[512];           // post: the saved x of the tile
    float lut[Q == 4 ? kWideCodes : Q == 2 ? kCodes : 1];
    double red[8];
};

// SOR: red-black passes, else damped-Jacobi sweeps; Q: 0 the FP32 channels, 2 / 4 one-byte / ten-bit codes
template <bool SOR, int Q, bool POST>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void dense_visit(TopoView tp, DenseArgs a,
                                                                                           const double* __restrict__ S)
{
    __shared__ DenseLds<Q> s;
    constexpr bool K = Q != 0;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // every wave holds the tile's row of the level's table, one word a lane
    const int tab = a.tab[size_t(kDenseWords) * blockIdx.x + lane];
    constexpr int TAB = K ? code_table<Q>() : 1;
    float lutv[K ? (TAB + 511) / 512 : 1];
    if constexpr (K) {
#pragma unroll
        for (int e = 0; e < (TAB + 511) / 512; ++e)
            lutv[e] = tid + 512 * e < TAB ? a.C.lut[size_t(a.level) * kWideCodes + tid + 512 * e] : 0.0f;
    }
    if (S[S_DONE] != 0.0) return;   // the solve has stopped (uniform)
    const int t = __builtin_amdgcn_readlane(tab, 13), nonleaf27 = __builtin_amdgcn_readlane(tab, kDenseNonleaf),
              oct = __builtin_amdgcn_readlane(tab, kDenseOct);
    const size_t base = size_t(t) * 512;
    const float h = tp.h0 / float(1 << a.level);
    const int passes = SOR ? 2 * a.iters : a.iters;
    const int deep = POST ? passes - 1 : passes;   // the deepest cells computed
    // the thread's cells, at region coordinates (0..15 are cells -4..11 of the tile) i, j and
    // j + 1, k..k+3: cell 4 r + e at (i, j + r, k + e).  The i of a wave have one parity, so
    // the colour of each cell is known without selects.
    const int i = 4 * (wave >> 1) + (wave & 1) + 2 * (lane >> 5), j = 2 * ((lane >> 2) & 7), q = lane & 3, k = 4 * q;
    const int odd = wave & 1;
    auto side = [](int r) { return r < 4 ? 0 : r < 12 ? 1 : 2; };
    auto depth = [](int r) { return r < 4 ? 4 - r : r > 11 ? r - 11 : 0; };
    auto cell_at = [](int ri, int rj, int rk) { return cidx((ri + 4) & 7, (rj + 4) & 7, (rk + 4) & 7); };
    // the least distance of the thread's cells from the tile
    const int dep = depth(i) + min(depth(j), depth(j + 1)) + ((q == 0 || q == 3) ? 1 : 0);
    const bool inner = dep == 0;   // cells of the tile
    const int n27 = 9 * side(i) + 3 * side(j) + side(k);
    const int tq = __shfl(tab, n27, 64);
    const int ti = __shfl(tab, 9 * side(i + 1) + 3 * side(j) + side(k), 64);
    const int tj = __shfl(tab, 9 * side(i) + 3 * side(j + 2) + side(k), 64);
    const int tk = __shfl(tab, 9 * side(i) + 3 * side(j) + side(k + 4), 64);
    const int tp27 = __shfl(tab, 27 + n27, 64);   // the parent of the cells' tile
    const bool nonleaf = (uint32_t(nonleaf27) >> n27) & 1u;
    const float* __restrict__ Xin = POST ? a.T : a.X;
    const float* __restrict__ Bin = POST && a.save ? a.BN : a.B;
    // the loads: x (and types) one cell deeper than the computed cells, the rest on those
    const bool here = tq >= 0 && dep <= deep, xin = tq >= 0 && dep <= deep + 1;
    float x[8] = {}, b[8] = {}, d[8] = {}, cm[8][3] = {}, cp0[8], cp1[4], ck[2] = {h, h};
    uint32_t ow[K ? 8 : 1] = {}, wi[K ? 8 : 1] = {}, wj[K ? 4 : 1] = {}, wk[2] = {};
    uint8_t ct[K ? 1 : 8] = {};
    float p1[2] = {}, p0[2] = {};
    auto row = [](auto& v, int r) -> auto& { return *reinterpret_cast<std::remove_reference_t<decltype(v[0])>(*)[4]>(&v[4 * r]); };
    if (xin) {
        const size_t v = size_t(tq) * 512 + cell_at(i, j, k);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            if (POST || !a.zero) vload<4>(Xin + v + 8 * r, row(x, r));
            if constexpr (K) vload<4>(a.C.w + v + 8 * r, row(ow, r));
            else vload<4>(tp.ctype + v + 8 * r, row(ct, r));
        }
        if constexpr (POST) {
            // the prolongation reads the parents' x and saved x
            const int bi = (oct + side(i) + 1) & 1, bj = ((oct >> 1) + side(j) + 1) & 1, bk = ((oct >> 2) + side(k) + 1) & 1;
            const size_t pv = size_t(tp27) * 512 +
                              cidx(4 * bi + (((i + 4) & 7) >> 1), 4 * bj + (((j + 4) & 7) >> 1), 4 * bk + (((k + 4) & 7) >> 1));
            vload<2>(a.X + pv, p1);
            vload<2>(a.X0 + pv, p0);
        }
    }
    if (here) {
        const size_t v = size_t(tq) * 512 + cell_at(i, j, k);
        const size_t vi = size_t(max(ti, 0)) * 512 + cell_at(i + 1, j, k), vj = size_t(max(tj, 0)) * 512 + cell_at(i, j + 2, k),
                     vk = size_t(max(tk, 0)) * 512 + cell_at(i, j, k + 4);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            vload<4>(Bin + v + 8 * r, row(b, r));
            vload<4>(a.C.c[3] + v + 8 * r, row(d, r));
        }
        if constexpr (K) {
            // (a missing neighbour tile: h, below)
#pragma unroll
            for (int r = 0; r < 2; ++r) vload<4>(a.C.w + vi + 8 * r, row(wi, r));
            vload<4>(a.C.w + vj, wj);
            if (q == 3) wk[0] = a.C.w[vk], wk[1] = a.C.w[vk + 8];
        } else {
            float c4[3][8];
#pragma unroll
            for (int f = 0; f < 3; ++f)
#pragma unroll
                for (int r = 0; r < 2; ++r) vload<4>(a.C.c[f] + v + 8 * r, row(c4[f], r));
#pragma unroll
            for (int r = 0; r < 2; ++r) vload<4>(a.C.c[0] + vi + 8 * r, row(cp0, r));
            vload<4>(a.C.c[1] + vj, cp1);
            ck[0] = a.C.c[2][vk];
            ck[1] = a.C.c[2][vk + 8];
#pragma unroll
            for (int c = 0; c < 8; ++c)
#pragma unroll
                for (int f = 0; f < 3; ++f) cm[c][f] = c4[f][c];
        }
    }
    // pre with four passes: x on the faces five cells out
    float sx = 0.0f;
    int sp = -1;
    if (!POST && deep == 4) {
        const int f = tid >> 6, fp = 4 + ((tid >> 3) & 7), fq = 4 + (tid & 7), axis = f >> 1, r = (f & 1) ? 16 : -1;
        const int ri = axis == 0 ? r : fp, rj = axis == 1 ? r : axis == 0 ? fp : fq, rk = axis == 2 ? r : fq;
        const int ts = __shfl(tab, 9 * side(ri) + 3 * side(rj) + side(rk), 64);
        if (tid < 384) {
            sp = (ri + 1) * kPlane + (rj + 1) * kRow + rk + 1;
            if (ts >= 0 && !a.zero) {
                const size_t v = size_t(ts) * 512 + cell_at(ri, rj, rk);
                uint8_t c;
                if constexpr (K) c = word_type<Q>(a.C.w[v]);
                else c = tp.ctype[v];
                const float xv = Xin[v];
                sx = c == INTERIOR ? xv : 0.0f;
            }
        }
    }
    if constexpr (K) {
#pragma unroll
        for (int e = 0; e < (TAB + 511) / 512; ++e)
            if (tid + 512 * e < TAB) s.lut[tid + 512 * e] = lutv[e];
        __syncthreads();
        // the word after the thread's cells along k is the next lane's (loaded by the last quad)
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const uint32_t nw = __shfl_down(ow[4 * r], 1, 64);
            wk[r] = q == 3 ? wk[r] : nw;
        }
    }
    // types, codes to values, x (the prolongation added) to LDS
    const int lx = (i + 1) * kPlane + (j + 1) * kRow + k + 1;
    uint32_t in = 0;   // bit c: cell c is INTERIOR
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        bool inc;
        if constexpr (K) {
            inc = word_type<Q>(ow[c]) & INTERIOR;   // (0 where nothing was loaded)
#pragma unroll
            for (int f = 0; f < 3; ++f) cm[c][f] = s.lut[word_code<Q>(ow[c], f)];
            cp0[c] = s.lut[word_code<Q>(wi[c], 0)];
            if (c < 4) cp1[c] = s.lut[word_code<Q>(wj[c], 1)];
        } else {
            inc = ct[c] & INTERIOR;
        }
        cp0[c] = ti < 0 ? h : cp0[c];
        if (c < 4) cp1[c] = tj < 0 ? h : cp1[c];
        in |= uint32_t(inc) << c;
        float v = x[c];
        if constexpr (POST) v = v + a.P * (p1[(c & 3) >> 1] - p0[(c & 3) >> 1]);
        x[c] = inc ? v : 0.0f;
        s.x[lx + (c >> 2) * kRow + (c & 3)] = x[c];
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        if constexpr (K) ck[r] = s.lut[word_code<Q>(wk[r], 2)];
        ck[r] = tk < 0 ? h : ck[r];
    }
    if (sp >= 0) s.x[sp] = sx;
    double rd[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) rd[c] = reciprocal(d[c]);
    // A x of a cell: the thread's own neighbours from registers, the others from LDS
    auto lap = [&](int c) {
        const int r = c >> 2, e = c & 3, l = lx + r * kRow + e;
        const float im = s.x[l - kPlane], ip = s.x[l + kPlane];
        const float jm = r ? x[e] : s.x[l - kRow], jp = r ? s.x[l + kRow] : x[4 + e];
        const float km = e ? x[c - (e ? 1 : 0)] : s.x[l - 1], kp = e < 3 ? x[c + (e < 3 ? 1 : 0)] : s.x[l + 1];
        float v = x[c] * d[c];
        v = fmaf(cm[c][0], im, v);
        v = fmaf(cp0[c], ip, v);
        v = fmaf(cm[c][1], jm, v);
        v = fmaf(r ? cp1[e] : cm[4 + e][1], jp, v);
        v = fmaf(cm[c][2], km, v);
        v = fmaf(e < 3 ? cm[c + (e < 3 ? 1 : 0)][2] : ck[r], kp, v);
        return d[c] == 0 ? 0.0f : v;
    };
    auto interior = [&](int c) { return (in >> c) & 1u; };
    const int ov = inner ? cell_at(i, j, k) : 0;   // the tile's cells: ov, ov + 8
    auto own_store = [&](float* p, float (&v)[8]) {
#pragma unroll
        for (int r = 0; r < 2; ++r) vstore<4>(p + ov + 8 * r, row(v, r));
    };
    __syncthreads();
    if (!POST && a.save) {
        // the FAS save of NONLEAF tiles: b += A x, the tile's own x saved
        if (nonleaf && dep <= deep) {
#pragma unroll
            for (int c = 0; c < 8; ++c) b[c] = interior(c) ? b[c] + lap(c) : 0.0f;
        }
        if (inner) {
            own_store(a.BN + base, b);
            if (nonleaf) {
#pragma unroll
                for (int c = 0; c < 8; ++c)
                    if (interior(c)) a.X0[base + ov + 8 * (c >> 2) + (c & 3)] = x[c];
            }
        }
        if (SOR) __syncthreads();   // every read of x for the save is done before x changes
    }
    if (POST && a.save && inner) own_store(a.B + base, b);
    // post: the fine row of this thread, for the prolongation into the level above
    const int fi = tid >> 5, fj = (tid >> 1) & 15, fk = tid & 1;
    int child = -1;
    uint8_t cty = 0;
    float px[8];
    uint8_t pc[8];
    if (POST && a.push) {
        const int32_t* cr = reinterpret_cast<const int32_t*>(a.rec + size_t(kRecWords) * blockIdx.x + 5);
        child = cr[(fi >> 3) | ((fj >> 3) << 1) | (fk << 2)];
        if (child >= 0) {
            const size_t fb = size_t(child) * 512 + cidx(fi & 7, fj & 7, 0);
            cty = tp.ttype[child];
            vload<8>(a.X + fb, px);
            vload<8>(tp.ctype + fb, pc);
        }
        s.v0[tid] = a.X0[base + tid];
    }
    double acc = 0;
    if constexpr (SOR) {
        // the thread's cells with r + e even (par 0) or odd
        auto half = [&](auto parity) {
            constexpr int par = decltype(parity)::value;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const int r = m >> 1, c = 4 * r + 2 * (m & 1) + (par ^ r);
                const float delta = interior(c) ? quotient(b[c] - lap(c), rd[c]) : 0.0f;
                x[c] = float(double(x[c]) + double(delta) * a.omega);
                s.x[lx + r * kRow + (c & 3)] = x[c];
            }
        };
        for (int p = 0; p < passes; ++p) {
            if (dep <= deep - p) {
                // pre: red first, post: black first
                if (((p & 1) ^ odd ^ int(POST)) == 0) half(std::integral_constant<int, 0>{});
                else half(std::integral_constant<int, 1>{});
            }
            __syncthreads();
        }
    } else {
        for (int p = 0; p < passes; ++p) {
            const bool go = dep <= deep - p;
            const bool zero = !POST && a.zero && p == 0;   // w b / d, also where a coefficient is not finite
            float xo[8];
            if (go) {
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    const float ax = lap(c);
                    const float delta = interior(c) ? quotient(b[c] - (zero ? 0.0f : ax), rd[c]) : 0.0f;
                    xo[c] = x[c] + a.w * delta;
                }
            }
            __syncthreads();   // every read of this sweep is done before x changes
            if (go) {
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    x[c] = interior(c) ? xo[c] : 0.0f;
                    s.x[lx + (c >> 2) * kRow + (c & 3)] = x[c];
                }
            }
            __syncthreads();
        }
    }
    if (inner) {
        own_store((POST ? a.X : a.T) + base, x);
        if constexpr (POST) {
            own_store(s.v, x);
            if (a.rz && !nonleaf) {
#pragma unroll
                for (int c = 0; c < 8; ++c) acc += double(b[c]) * double(x[c]);
            }
        } else {
            float r8[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) r8[c] = b[c] - lap(c);
            own_store(s.v, r8);
        }
    }
    if constexpr (!POST) {
        __syncthreads();
        if (tid >= 64) return;
        const int pt = __builtin_amdgcn_readlane(tab, 27 + 13);
        const int fl0 = tid / 16 * 2, fl1 = (tid / 4) % 4 * 2, fl2 = tid % 4 * 2;
        float rs = 0, xs = 0;
#pragma unroll
        for (int ii = 0; ii < 2; ++ii)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                for (int kk = 0; kk < 2; ++kk) {
                    rs += s.v[cidx(fl0 + ii, fl1 + jj, fl2 + kk)];
                    xs += s.x[(fl0 + ii + 5) * kPlane + (fl1 + jj + 5) * kRow + fl2 + kk + 5];
                }
        const size_t pidx = size_t(pt) * 512 + cidx(4 * (oct & 1) + (fl0 >> 1), 4 * ((oct >> 1) & 1) + (fl1 >> 1),
                                                    4 * ((oct >> 2) & 1) + (fl2 >> 1));
        a.B[pidx] = rs * a.Rr;
        a.X[pidx] = xs / 8;
    } else {
        if (a.push) {
            __syncthreads();
            if (child >= 0) {
                const int pv = cidx(fi >> 1, fj >> 1, 4 * fk);
                const bool ghost = cty & GHOST;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const bool inf = pc[e] & INTERIOR;
                    const float c1 = s.v[pv + (e >> 1)], c0 = s.v0[pv + (e >> 1)];
                    px[e] = ghost ? (inf ? c1 : 0.0f) : (inf ? px[e] + a.P * (c1 - c0) : 0.0f);
                }
                vstore<8>(a.X + size_t(child) * 512 + cidx(fi & 7, fj & 7, 0), px);
            }
        }
        if (a.rz) {
            const double sum = block_sum(acc, s.red);
            if (tid == 0) a.rz[blockIdx.x] = sum;
        }
    }
}

}  // namespace k

template <bool SOR, bool POST>
static void dense_launch(const DevGrid& d, int n, int form, const k::DenseArgs& a, const double* S, hipStream_t st)
{
    const TopoView tp = view(d);
    switch (form) {
    case 2: k::dense_visit<SOR, 2, POST><<<n, 512, 0, st>>>(tp, a, S); break;
    case 4: k::dense_visit<SOR, 4, POST><<<n, 512, 0, st>>>(tp, a, S); break;
    default: k::dense_visit<SOR, 0, POST><<<n, 512, 0, st>>>(tp, a, S); break;
    }
}

// four passes are what the 16^3 cells hold (the residual needs one cell more).  Jacobi with three and four sweeps,
// eight iterations with a V-cycle, a launch a pass against this: uniform 64^3 955 -> 766 us and 997 -> 821 us, the
// 256^3 sphere 2,408 -> 2,177 and 2,590 -> 2,403 (two sweeps: the figures above)
bool dense_visit_fits(bool rbgs, int iters) { return iters >= 1 && iters <= (rbgs ? 2 : 4); }

void launch_dense_visit(const DevGrid& d, int level, bool post, float* X, float* T, float* B, float* BN, float* X0, Coef C,
                        float Rr, float P, bool rbgs, int iters, double omega, bool zero, bool save, bool push, double* rz,
                        const double* S, hipStream_t st)
{
    const LaunchList& l = d.subtree[level];
    if (level < 1 || !d.dense[level] || C.q[0] || !dense_visit_fits(rbgs, iters) || (push && !d.push_ok[level + 1]))
        throw std::logic_error("dense_visit: the level or the settings do not fit");
    k::DenseArgs a;
    a.tab = d.dense[level];
    a.rec = l.rec;
    a.X = X; a.T = T; a.B = B; a.BN = BN; a.X0 = X0; a.C = C;
    a.Rr = Rr; a.P = P; a.w = float(omega); a.omega = omega;
    a.level = level; a.iters = iters; a.zero = zero; a.save = save; a.push = push; a.rz = rz;
    const int form = C.w && ((C.coded >> level) & 1u) ? (((C.wide >> level) & 1u) ? 4 : 2) : 0;
    const double* Sr = S ? S : d.idle;
    if (rbgs && post) dense_launch<true, true>(d, l.n, form, a, Sr, st);
    else if (rbgs) dense_launch<true, false>(d, l.n, form, a, Sr, st);
    else if (post) dense_launch<false, true>(d, l.n, form, a, Sr, st);
    else dense_launch<false, false>(d, l.n, form, a, Sr, st);
}

}  // namespace cmg
