// cmg_geo.hip -- gfx950 kernels of the two geometric multigrid solvers:
// GMGSolver (src/GMGSolver.cu) and CMGSolver (src/CMGSolver.cu).
//
// Both operators come from cell and tile types alone:
//   GMG  face coefficient (1/dh)(1/h): dh = h between LEAF cells, 1.5 h
//        between a LEAF and a GHOST cell, else 0; 0 next to a NEUMANN cell;
//        the cell sum is scaled by h^3 (GMGSolver.cu:3-67)
//   CMG  face coefficient h, 0 next to a NEUMANN cell; GHOST neighbours are
//        extrapolated as in the AMG loader (CMGSolver.cu:3-170)
// One 8^3 tile per 256-thread workgroup; x (unmasked) and the cell types are
// staged in LDS.  Arithmetic is written out
// (fp-contract off, explicit fmaf) so that results match the CPU restatement
// bit for bit:  sum = fmaf(c, x0 - x1, sum) over axis 0..2, side -,+.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdexcept>
#include <type_traits>

#include "cmg_device.hpp"
#include "cmg_kernels.hpp"

#pragma clang fp contract(off)

namespace cmg {
namespace k {

constexpr int GEO_GMG = 0, GEO_CMG = 1;

struct GeoLds {
    float x[1000];
    uint8_t ct[1000];
};

// HATileInfo::subtreeType (src/HATileInfo.h:79-84); subtree_level < 0: the own type
__device__ __forceinline__ uint8_t subtree_type(uint8_t type, int level, int subtree_level)
{
    return (level == subtree_level && type == NONLEAF) ? uint8_t(LEAF) : type;
}

// NegativeLaplacianCoeff (GMGSolver.cu:3-30 / CMGSolver.cu:3-7) between two cells that are not NEUMANN
template <int MODE>
__device__ __forceinline__ float geo_open_coeff(float h, float one_over_h, uint8_t t0, uint8_t t1)
{
    if (MODE == GEO_CMG) return h;
    const bool both = (t0 & LEAF) && (t1 & LEAF);
    const bool lg = ((t0 & LEAF) && (t1 & GHOST)) || ((t0 & GHOST) && (t1 & LEAF));
    const float odh = both ? one_over_h : lg ? (2 * one_over_h / 3) : 0.0f;
    return odh * one_over_h;
}

// A tile's open-face coefficients: inside it and behind its faces (x-, x+, y-, y+, z-, z+)
struct GeoTile {
    float h, in, face[6];
    uint8_t own;   // subtree type
};

// LoadGMGLaplacianTileData (GMGSolver.cu:81-133) / LoadCMGLaplacianTileData (CMGSolver.cu:62-170).
// The tile's record (scalar loads) gives every address and face coefficient, so the tile's
// cells and its halo are one round trip; only CMG's ghost extrapolation waits for the tile's
// own values.  256 threads, two cells (v0, v0 + 1) along k each.
template <int MODE>
__device__ __forceinline__ GeoTile geo_load(const TopoView& tp, const TileRec& r, int subtree_level, const float* __restrict__ X,
                                            GeoLds& s)
{
    const int tid = threadIdx.x, v0 = 2 * tid;
    const size_t base = size_t(r.t) * 512;
    const uint32_t ty03 = uint32_t(r.hb.z), ty45 = uint32_t(r.hb.w);
    GeoTile g;
    g.h = rec_h(tp, r);
    g.own = subtree_type(uint8_t(r.meta & 0xff), r.level, subtree_level);
    float xo[2];
    uint8_t co[2];
    vload<2>(X + base + v0, xo);
    vload<2>(tp.ctype + base + v0, co);
    // halo: face f = 2 axis + (side > 0) of elements 64 f .. 64 f + 63 (the tile's own cells where it has no neighbour)
    float xn[2];
    uint8_t cn[2];
    int at[2], cl[2];   // halo cell in LDS, the tile's cell next to it
    bool ghost[2], none[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        const int e = min(tid + 256 * m, 383), f = e >> 6, fi = e & 63;
        const int axis = f >> 1, sgn = (f & 1) ? 1 : -1, slot = sgn < 0 ? axis : axis + 3;
        const int p = fi >> 3, q = fi & 7, lo = sgn < 0 ? 7 : 0, ax = sgn < 0 ? -1 : 8;
        const int a0 = axis == 0 ? ax : p, a1 = axis == 1 ? ax : axis == 0 ? p : q, a2 = axis == 2 ? ax : q;
        const int nt = pick6(r.ha, r.hb, slot);
        const size_t ni = size_t(nt >= 0 ? nt : r.t) * 512 + cidx(axis == 0 ? lo : a0, axis == 1 ? lo : a1, axis == 2 ? lo : a2);
        xn[m] = X[ni];
        cn[m] = tp.ctype[ni];
        at[m] = SX(a0, a1, a2);
        cl[m] = cidx(a0 - (axis == 0 ? sgn : 0), a1 - (axis == 1 ? sgn : 0), a2 - (axis == 2 ? sgn : 0));
        none[m] = nt < 0;
        ghost[m] = nt >= 0 && ((slot < 4 ? ty03 >> (8 * slot) : ty45 >> (8 * (slot - 4))) & GHOST);
    }
    // the face coefficients (uniform over the workgroup)
    const float one_over_h = 1 / g.h;
    g.in = geo_open_coeff<MODE>(g.h, one_over_h, g.own, g.own);
    const int nb[6] = {r.ha.x, r.ha.w, r.ha.y, r.hb.x, r.ha.z, r.hb.y};
    const uint32_t ty[6] = {ty03, ty03 >> 24, ty03 >> 8, ty45, ty03 >> 16, ty45 >> 8};
#pragma unroll
    for (int f = 0; f < 6; ++f)
        g.face[f] = geo_open_coeff<MODE>(g.h, one_over_h, g.own,
                                         nb[f] < 0 ? g.own : subtree_type(uint8_t(ty[f]), r.level, subtree_level));
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int l = SX(v0 >> 6, (v0 >> 3) & 7, (v0 & 7) + c);
        s.x[l] = xo[c];
        s.ct[l] = co[c];
    }
    if constexpr (MODE == GEO_CMG) __syncthreads();
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        if (m == 1 && tid >= 128) continue;
        float xv = none[m] ? 0.0f : xn[m];
        if (MODE == GEO_CMG && ghost[m]) {
            float avg = 0;
#pragma unroll
            for (int di = 0; di < 2; ++di)
#pragma unroll
                for (int dj = 0; dj < 2; ++dj)
#pragma unroll
                    for (int dk = 0; dk < 2; ++dk) {
                        const int b = cl[m] ^ ((di << 6) | (dj << 3) | dk);
                        avg += s.x[SX(b >> 6, (b >> 3) & 7, b & 7)];
                    }
            avg /= 8;
            xv = float(double(s.x[SX(cl[m] >> 6, (cl[m] >> 3) & 7, cl[m] & 7)]) + 0.5 * double(xn[m] - avg));
        }
        s.x[at[m]] = xv;
        s.ct[at[m]] = none[m] ? uint8_t(DIRICHLET) : cn[m];
    }
    __syncthreads();
    return g;
}

// GMGLaplacianTileData::negativeLap (GMGSolver.cu:45-66) / CMG (CMGSolver.cu:23-45) of cell v, and
// (diag) the sum of its coefficients
template <int MODE>
__device__ __forceinline__ float geo_neg_lap(const GeoLds& s, const GeoTile& g, int v, float& diag)
{
    const int l[3] = {v >> 6, (v >> 3) & 7, v & 7};
    const int c = SX(l[0], l[1], l[2]);
    const uint8_t c0 = s.ct[c];
    const float x0 = s.x[c];
    const int step[3] = {100, 10, 1};
    float sum = 0, dg = 0;
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        const int a = f >> 1, n = c + ((f & 1) ? step[a] : -step[a]);
        const bool inside = (f & 1) ? l[a] < 7 : l[a] > 0;
        const float k = ((c0 | s.ct[n]) & NEUMANN) ? 0.0f : inside ? g.in : g.face[f];
        dg = dg + k;
        sum = fmaf(k, x0 - s.x[n], sum);
    }
    const float h = g.h;
    diag = !(c0 & INTERIOR) ? 0.0f : MODE == GEO_GMG ? dg * h * h * h : dg;
    return !(c0 & INTERIOR) ? 0.0f : MODE == GEO_GMG ? sum * h * h * h : sum;
}

// NegativeLaplacianSameLevel128Kernel (GMGSolver.cu:135-161) / CMG twin (CMGSolver.cu:172-201)
template <int MODE>
__global__ __launch_bounds__(256) void geo_apply(TopoView tp, const int4* __restrict__ rec, int subtree_level,
                                                 const float* __restrict__ X, float* __restrict__ Y, int diag,
                                                 const double* __restrict__ S)
{
    __shared__ GeoLds s;
    const TileRec r = rec_tile<false>(rec, S);
    if (r.t < 0) return;   // no tile, or the solve has stopped
    const GeoTile g = geo_load<MODE>(tp, r, subtree_level, X, s);
    const int v0 = 2 * int(threadIdx.x);
    float y[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        float d;
        const float ax = geo_neg_lap<MODE>(s, g, v0 + c, d);
        y[c] = diag ? d : ax;
    }
    vstore<2>(Y + size_t(r.t) * 512 + v0, y);
}

// one colour of NegativeLaplacianAndGaussSeidelSameLevel128Kernel (GMGSolver.cu:173-206 / CMGSolver.cu:228-264):
// of a thread's two cells the one of that colour.  Latency and
// instruction issue bound it more than its 13 B a cell: one cell a thread, every colour's
// cells computed and the halo's addresses read through two dependent loads took 17.5 us for
// 4,672 tiles, this takes 10.3 us (MI355X, GMG; the operator 33.2 to 18.5 us).
template <int MODE>
__global__ __launch_bounds__(256) void geo_gs(TopoView tp, const int4* __restrict__ rec, int level, float* __restrict__ X,
                                              const float* __restrict__ B, int color, const double* __restrict__ S)
{
    __shared__ GeoLds s;
    const TileRec r = rec_tile<false>(rec, S);
    if (r.t < 0) return;   // no tile, or the solve has stopped
    const int v0 = 2 * int(threadIdx.x), v = v0 + (((v0 >> 6) + ((v0 >> 3) & 7) + color) & 1);
    const size_t idx = size_t(r.t) * 512 + v;
    const float b = B[idx];
    const GeoTile g = geo_load<MODE>(tp, r, level, X, s);
    const int c = SX(v >> 6, (v >> 3) & 7, v & 7);
    float d;
    const float ax = geo_neg_lap<MODE>(s, g, v, d);
    const float delta = (s.ct[c] & INTERIOR) ? (b - ax) / d : 0.0f;
    X[idx] = s.x[c] + delta;
}

// ResidualAndRestrict128Kernel (GMGSolver.cu:215-275) / CMG twin (CMGSolver.cu:273-330):
// parent b = sum8 r * one_over_alpha; a GHOST tile (GMG) adds sum8 r to its parent
template <int MODE>
__global__ __launch_bounds__(256) void geo_restrict(TopoView tp, const int4* __restrict__ rec, int level,
                                                    const float* __restrict__ X, float* __restrict__ B, float one_over_alpha,
                                                    const double* __restrict__ S)
{
    __shared__ GeoLds s;
    __shared__ float res[512];
    const TileRec r = rec_tile<false>(rec, S);
    if (r.t < 0) return;   // no tile, or the solve has stopped
    const int v = threadIdx.x;
    float b[2];
    vload<2>(B + size_t(r.t) * 512 + 2 * v, b);
    const GeoTile g = geo_load<MODE>(tp, r, level, X, s);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        float d;
        b[c] = b[c] - geo_neg_lap<MODE>(s, g, 2 * v + c, d);
    }
    vstore<2>(&res[2 * v], b);
    __syncthreads();
    if (v >= 64) return;
    const int pt = r.parent;
    if (pt < 0) return;
    const int oc = (r.meta >> 8) & 7;
    const int fl0 = v / 16 * 2, fl1 = (v / 4) % 4 * 2, fl2 = v % 4 * 2;
    float sum = 0;
#pragma unroll
    for (int ii = 0; ii < 2; ++ii)
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) sum += res[cidx(fl0 + ii, fl1 + jj, fl2 + kk)];
    const size_t pidx =
        size_t(pt) * 512 + cidx(4 * (oc & 1) + (fl0 >> 1), 4 * ((oc >> 1) & 1) + (fl1 >> 1), 4 * ((oc >> 2) & 1) + (fl2 >> 1));
    if (g.own & GHOST) B[pidx] = B[pidx] + sum;
    else B[pidx] = sum * one_over_alpha;
}

// Face coefficients and diagonals where every cell of the neighbourhood belongs to the level (no
// GHOST tile): an open face has geo_open_coeff's value K, one next to a NEUMANN cell 0, so a cell's
// coefficients are six bits and its diagonal one of seven values.
template <int MODE>
__device__ __forceinline__ float geo_face(float h)
{
    const float one_over_h = 1 / h;
    return MODE == GEO_CMG ? h : one_over_h * one_over_h;
}
template <int MODE>
__device__ __forceinline__ float geo_diag(float h, int faces)
{
    float sum = 0;
    for (int f = 0; f < faces; ++f) sum = sum + geo_face<MODE>(h);
    return MODE == GEO_GMG ? sum * h * h * h : sum;
}
// geo_neg_lap of an INTERIOR cell with value x0 from the neighbour values in its order
template <int MODE>
__device__ __forceinline__ float geo_lap6(float h, float K, uint32_t open, float x0, const float (&n)[6])
{
    float sum = 0;
#pragma unroll
    for (int f = 0; f < 6; ++f) sum = fmaf((open >> f) & 1u ? K : 0.0f, x0 - n[f], sum);
    return MODE == GEO_GMG ? sum * h * h * h : sum;
}

// A V-cycle's visit to a complete level (DevGrid::dense) in two launches, as dense_visit does
// it for the AMG cycles: a workgroup takes its tile with a halo as deep as the passes and
// computes the halo's cells again, so no pass waits for the neighbours.  POST false: the
// red-black iterations from x = 0 (x into T), the residual and its restriction into B below;
// true: the prolongation (prolong_add_v) onto T, the iterations from black, x into X.  The
// operations are those of geo_gs, geo_restrict and prolong_add_v, with quotient() in the place
// of the division.  At most two iterations.
// Bound by launch latency before (ten launches of about 4 us a visit) and by the issue of the
// halo's work now: MI355X, GMG, 11.3 + 10.7 us a visit to 512 tiles, 7.9 + 7.0 us to 64.
constexpr int kGeoRow = 21, kGeoPlane = 18 * kGeoRow;   // x in LDS, see cmg_dense.hip

template <int MODE, bool POST>
__global__ __launch_bounds__(512) void geo_dense(TopoView tp, const int32_t* __restrict__ table, int level, int iters,
                                                 float* __restrict__ X, float* __restrict__ T, float* __restrict__ B,
                                                 float one_over_alpha, float P, const double* __restrict__ S)
{
    __shared__ float sx[18 * kGeoPlane];
    __shared__ uint8_t sc[18 * kGeoPlane];
    __shared__ float res[512];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tab = table[size_t(kDenseWords) * blockIdx.x + lane];
    if (S[S_DONE] != 0.0) return;   // the solve has stopped (uniform)
    const int t = __builtin_amdgcn_readlane(tab, 13), oct = __builtin_amdgcn_readlane(tab, kDenseOct);
    const float h = tp.h0 / float(1 << level), K = geo_face<MODE>(h);
    const int passes = 2 * iters, deep = POST ? passes - 1 : passes;
    // the thread's cells, at region coordinates (0..15 are cells -4..11 of the tile) i, j and
    // j + 1, k..k+3: cell 4 r + e at (i, j + r, k + e); the i of a wave have one parity
    const int i = 4 * (wave >> 1) + (wave & 1) + 2 * (lane >> 5), j = 2 * ((lane >> 2) & 7), q = lane & 3, k = 4 * q;
    const int odd = wave & 1;
    auto side = [](int r) { return r < 4 ? 0 : r < 12 ? 1 : 2; };
    auto depth = [](int r) { return r < 4 ? 4 - r : r > 11 ? r - 11 : 0; };
    auto cell_at = [](int ri, int rj, int rk) { return cidx((ri + 4) & 7, (rj + 4) & 7, (rk + 4) & 7); };
    const int dep = depth(i) + min(depth(j), depth(j + 1)) + ((q == 0 || q == 3) ? 1 : 0);
    const bool inner = dep == 0;
    const int n27 = 9 * side(i) + 3 * side(j) + side(k);
    const int tq = __shfl(tab, n27, 64), pq = __shfl(tab, 27 + n27, 64);
    const bool here = tq >= 0 && dep <= deep, near = tq >= 0 && dep <= deep + 1;
    float x[8] = {}, b[8] = {};
    uint8_t ct[8] = {};
    float px[2] = {};
    auto row = [](auto& v, int r) -> auto& { return *reinterpret_cast<std::remove_reference_t<decltype(v[0])>(*)[4]>(&v[4 * r]); };
    if (near) {
        const size_t v = size_t(tq) * 512 + cell_at(i, j, k);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            vload<4>(tp.ctype + v + 8 * r, row(ct, r));
            if (POST) vload<4>(T + v + 8 * r, row(x, r));
        }
        if (POST) {
            const int bi = (oct + side(i) + 1) & 1, bj = ((oct >> 1) + side(j) + 1) & 1, bk = ((oct >> 2) + side(k) + 1) & 1;
            vload<2>(X + size_t(pq) * 512 + cidx(4 * bi + (((i + 4) & 7) >> 1), 4 * bj + (((j + 4) & 7) >> 1), 4 * bk + (((k + 4) & 7) >> 1)),
                     px);
        }
    }
    if (here) {
        const size_t v = size_t(tq) * 512 + cell_at(i, j, k);
#pragma unroll
        for (int r = 0; r < 2; ++r) vload<4>(B + v + 8 * r, row(b, r));
    }
    // the types of the faces five cells out (four passes); a cell without tile is DIRICHLET
    uint8_t sct = DIRICHLET;
    int sp = -1;
    if (deep == 4) {
        const int f = tid >> 6, fp = 4 + ((tid >> 3) & 7), fq = 4 + (tid & 7), axis = f >> 1, r = (f & 1) ? 16 : -1;
        const int ri = axis == 0 ? r : fp, rj = axis == 1 ? r : axis == 0 ? fp : fq, rk = axis == 2 ? r : fq;
        const int ts = __shfl(tab, 9 * side(ri) + 3 * side(rj) + side(rk), 64);
        if (tid < 384) {
            sp = (ri + 1) * kGeoPlane + (rj + 1) * kGeoRow + rk + 1;
            if (ts >= 0) sct = tp.ctype[size_t(ts) * 512 + cell_at(ri, rj, rk)];
        }
    }
    for (int e = tid; e < 18 * kGeoPlane; e += 512) sx[e] = 0.0f;
    __syncthreads();
    const int lx = (i + 1) * kGeoPlane + (j + 1) * kGeoRow + k + 1;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int l = lx + (c >> 2) * kGeoRow + (c & 3);
        if (POST) {
            x[c] = (ct[c] & INTERIOR) ? x[c] + P * px[(c & 3) >> 1] : 0.0f;
            sx[l] = x[c];
        }
        sc[l] = tq >= 0 ? ct[c] : uint8_t(DIRICHLET);
    }
    if (sp >= 0) sc[sp] = sct;
    __syncthreads();
    // open faces (x-, x+, y-, y+, z-, z+) six bits a cell, diagonals by their number
    uint32_t in = 0;
    uint64_t open = 0;
    double rd[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int l = lx + (c >> 2) * kGeoRow + (c & 3);
        const int nb[6] = {l - kGeoPlane, l + kGeoPlane, l - kGeoRow, l + kGeoRow, l - 1, l + 1};
        uint32_t o = 0;
#pragma unroll
        for (int f = 0; f < 6; ++f) o |= uint32_t(((ct[c] | sc[nb[f]]) & NEUMANN) == 0) << f;
        open |= uint64_t(o) << (6 * c);
        in |= uint32_t((ct[c] & INTERIOR) != 0) << c;
        const int m = __popc(o);
        float d = 0;
#pragma unroll
        for (int f = 0; f < 6; ++f) d = f < m ? d + K : d;
        if (MODE == GEO_GMG) d = d * h * h * h;
        rd[c] = reciprocal(d);
    }
    auto lap = [&](int c) {
        const int r = c >> 2, e = c & 3, l = lx + r * kGeoRow + e;
        const float n[6] = {sx[l - kGeoPlane], sx[l + kGeoPlane], r ? x[e] : sx[l - kGeoRow], r ? sx[l + kGeoRow] : x[4 + e],
                            e ? x[c - (e ? 1 : 0)] : sx[l - 1], e < 3 ? x[c + (e < 3 ? 1 : 0)] : sx[l + 1]};
        return (in >> c) & 1u ? geo_lap6<MODE>(h, K, uint32_t(open >> (6 * c)), x[c], n) : 0.0f;
    };
    auto half = [&](auto parity) {
        constexpr int par = decltype(parity)::value;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const int r = m >> 1, c = 4 * r + 2 * (m & 1) + (par ^ r);
            const float delta = (in >> c) & 1u ? quotient(b[c] - lap(c), rd[c]) : 0.0f;
            x[c] = x[c] + delta;
            sx[lx + r * kGeoRow + (c & 3)] = x[c];
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
    const int ov = inner ? cell_at(i, j, k) : 0;
    if (inner) {
#pragma unroll
        for (int r = 0; r < 2; ++r) vstore<4>((POST ? X : T) + size_t(t) * 512 + ov + 8 * r, row(x, r));
        if (!POST) {
            float v[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) v[c] = b[c] - lap(c);
#pragma unroll
            for (int r = 0; r < 2; ++r) vstore<4>(&res[ov + 8 * r], row(v, r));
        }
    }
    if (POST) return;
    __syncthreads();
    if (tid >= 64) return;
    const int fl0 = tid / 16 * 2, fl1 = (tid / 4) % 4 * 2, fl2 = tid % 4 * 2;
    float sum = 0;
#pragma unroll
    for (int ii = 0; ii < 2; ++ii)
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) sum += res[cidx(fl0 + ii, fl1 + jj, fl2 + kk)];
    const int pt = __builtin_amdgcn_readlane(tab, 27 + 13);
    B[size_t(pt) * 512 + cidx(4 * (oct & 1) + (fl0 >> 1), 4 * ((oct >> 1) & 1) + (fl1 >> 1), 4 * ((oct >> 2) & 1) + (fl2 >> 1))] =
        sum * one_over_alpha;
}

// the iterations on a level 0 of one tile without neighbours, in one workgroup: `iters` from
// red, then `iters` from black, two cells a thread (one of each colour) with x in LDS.  (MI355X,
// 10 coarsest iterations: 5.3 us against 20 launches of 3 us.)
template <int MODE>
__global__ __launch_bounds__(256) void geo_root(TopoView tp, int t, int iters, float* __restrict__ X, const float* __restrict__ B,
                                                const double* __restrict__ S)
{
    __shared__ float sx[1000];
    __shared__ uint8_t sc[1000];
    if (S[S_DONE] != 0.0) return;   // the solve has stopped (uniform)
    const int tid = threadIdx.x, i = tid >> 5, j = (tid >> 2) & 7, k = 2 * (tid & 3);
    const bool odd = (i + j) & 1;
    const float h = tp.h0, K = geo_face<MODE>(h);
    const size_t v0 = size_t(t) * 512 + cidx(i, j, k);
    float xv[2], bv[2];
    uint8_t cv[2];
    vload<2>(X + v0, xv);
    vload<2>(B + v0, bv);
    vload<2>(tp.ctype + v0, cv);
    for (int e = tid; e < 1000; e += 256) {
        sx[e] = 0.0f;
        sc[e] = DIRICHLET;
    }
    __syncthreads();
    // [0] the red cell, [1] the black one
    const int l[2] = {SX(i, j, k + int(odd)), SX(i, j, k + 1 - int(odd))};
    float x[2], b[2];
    uint8_t ct[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const bool second = bool(e) != odd;
        x[e] = second ? xv[1] : xv[0];
        b[e] = second ? bv[1] : bv[0];
        ct[e] = second ? cv[1] : cv[0];
        sx[l[e]] = x[e];
        sc[l[e]] = ct[e];
    }
    __syncthreads();
    uint32_t open[2];
    double rd[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int nb[6] = {l[e] - 100, l[e] + 100, l[e] - 10, l[e] + 10, l[e] - 1, l[e] + 1};
        open[e] = 0;
#pragma unroll
        for (int f = 0; f < 6; ++f) open[e] |= uint32_t(((ct[e] | sc[nb[f]]) & NEUMANN) == 0) << f;
        rd[e] = reciprocal(geo_diag<MODE>(h, __popc(open[e])));
    }
    auto pass = [&](auto colour) {
        constexpr int e = decltype(colour)::value;
        const float n[6] = {sx[l[e] - 100], sx[l[e] + 100], sx[l[e] - 10], sx[l[e] + 10], sx[l[e] - 1], sx[l[e] + 1]};
        const bool in = ct[e] & INTERIOR;
        const float ax = in ? geo_lap6<MODE>(h, K, open[e], x[e], n) : 0.0f;
        x[e] = x[e] + (in ? quotient(b[e] - ax, rd[e]) : 0.0f);
        sx[l[e]] = x[e];
        __syncthreads();
    };
    using Red = std::integral_constant<int, 0>;
    using Black = std::integral_constant<int, 1>;
    for (int it = 0; it < iters; ++it) {
        pass(Red{});
        pass(Black{});
    }
    for (int it = 0; it < iters; ++it) {
        pass(Black{});
        pass(Red{});
    }
    X[v0 + int(odd)] = x[0];
    X[v0 + 1 - int(odd)] = x[1];
}

// AccumulateToParentsOneStep(GHOST, coeff, additive, all cell types) (src/PoissonGrid.cu:408-465)
__global__ __launch_bounds__(64) void accumulate_add(TopoView tp, const int32_t* __restrict__ list, float* __restrict__ Y,
                                                     float coeff, const double* __restrict__ S)
{
    if (stopped(S)) return;
    const int t = list[blockIdx.x];
    if (t < 0) return;
    const int pt = tp.parent[t];
    if (pt < 0) return;
    const int v = threadIdx.x, oc = tp.toct[t];
    const int fl0 = v / 16 * 2, fl1 = (v / 4) % 4 * 2, fl2 = v % 4 * 2;
    float sum = 0;
#pragma unroll
    for (int ii = 0; ii < 2; ++ii)
#pragma unroll
        for (int jj = 0; jj < 2; ++jj)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) sum += Y[size_t(t) * 512 + cidx(fl0 + ii, fl1 + jj, fl2 + kk)];
    const size_t pidx =
        size_t(pt) * 512 + cidx(4 * (oc & 1) + (fl0 >> 1), 4 * ((oc >> 1) & 1) + (fl1 >> 1), 4 * ((oc >> 2) & 1) + (fl2 >> 1));
    Y[pidx] = Y[pidx] + sum * coeff;
}

// r = b - Ax on INTERIOR cells of LEAF tiles, Ax kept elsewhere (GMGSolver.cu:421-431)
__global__ __launch_bounds__(256) void residual_interior_v(TopoView tp, const int32_t* __restrict__ list, int n,
                                                           const float* __restrict__ B, float* __restrict__ AX)
{
    CMG_TILE_LOOP(list, n)
    {
        const size_t q = quad_index(t_);
        const uchar4 ct = reinterpret_cast<const uchar4*>(tp.ctype)[q];
        const float4 b = reinterpret_cast<const float4*>(B)[q];
        float4 a = reinterpret_cast<const float4*>(AX)[q];
        if (ct.x & INTERIOR) a.x = b.x - a.x;
        if (ct.y & INTERIOR) a.y = b.y - a.y;
        if (ct.z & INTERIOR) a.z = b.z - a.z;
        if (ct.w & INTERIOR) a.w = b.w - a.w;
        reinterpret_cast<float4*>(AX)[q] = a;
    }
}

// damped-Jacobi update x += omega r / D on INTERIOR cells, x = 0 where D = 0 (GMGSolver.cu:448-466)
__global__ __launch_bounds__(256) void djacobi_update_v(TopoView tp, const int32_t* __restrict__ list, int n,
                                                        float* __restrict__ X, const float* __restrict__ R,
                                                        const float* __restrict__ D, float omega)
{
    CMG_TILE_LOOP(list, n)
    {
        const size_t q = quad_index(t_);
        const uchar4 ct = reinterpret_cast<const uchar4*>(tp.ctype)[q];
        const float4 r = reinterpret_cast<const float4*>(R)[q];
        const float4 d = reinterpret_cast<const float4*>(D)[q];
        float4 x = reinterpret_cast<const float4*>(X)[q];
        if (ct.x & INTERIOR) x.x = d.x == 0 ? 0.0f : x.x + omega * r.x / d.x;
        if (ct.y & INTERIOR) x.y = d.y == 0 ? 0.0f : x.y + omega * r.y / d.y;
        if (ct.z & INTERIOR) x.z = d.z == 0 ? 0.0f : x.z + omega * r.z / d.z;
        if (ct.w & INTERIOR) x.w = d.w == 0 ? 0.0f : x.w + omega * r.w / d.w;
        reinterpret_cast<float4*>(X)[q] = x;
    }
}

}  // namespace k

// ---------------------------------------------------------------- launchers ---

static inline int geo_vector_grid(const DevGrid& d, int n) { return std::max(1, std::min((n + 1) / 2, d.wg_cap)); }

void launch_geo_apply(const DevGrid& d, int mode, const LaunchList& l, int subtree_level, const float* X, float* Y, bool diag,
                      const double* S, hipStream_t st)
{
    if (l.n <= 0) return;
    if (mode == k::GEO_GMG) k::geo_apply<k::GEO_GMG><<<l.n, 256, 0, st>>>(view(d), l.rec, subtree_level, X, Y, int(diag), S ? S : d.idle);
    else k::geo_apply<k::GEO_CMG><<<l.n, 256, 0, st>>>(view(d), l.rec, subtree_level, X, Y, int(diag), S ? S : d.idle);
}

void launch_geo_gs(const DevGrid& d, int mode, int level, float* X, const float* B, int color, const double* S, hipStream_t st)
{
    const LaunchList& l = d.subtree[level];
    if (l.n <= 0) return;
    if (mode == k::GEO_GMG) k::geo_gs<k::GEO_GMG><<<l.n, 256, 0, st>>>(view(d), l.rec, level, X, B, color, S ? S : d.idle);
    else k::geo_gs<k::GEO_CMG><<<l.n, 256, 0, st>>>(view(d), l.rec, level, X, B, color, S ? S : d.idle);
}

void launch_geo_restrict(const DevGrid& d, int mode, int level, const float* X, float* B, float one_over_alpha,
                         const double* S, hipStream_t st)
{
    // GMG restricts from every tile of the level (GHOST included), CMG from LEAF|NONLEAF tiles
    const LaunchList& l = mode == k::GEO_GMG ? d.prolong[level] : d.subtree[level];
    if (l.n <= 0) return;
    if (mode == k::GEO_GMG) k::geo_restrict<k::GEO_GMG><<<l.n, 256, 0, st>>>(view(d), l.rec, level, X, B, one_over_alpha, S ? S : d.idle);
    else k::geo_restrict<k::GEO_CMG><<<l.n, 256, 0, st>>>(view(d), l.rec, level, X, B, one_over_alpha, S ? S : d.idle);
}

void launch_geo_dense(const DevGrid& d, int mode, int level, bool post, int iters, float* X, float* T, float* B,
                      float one_over_alpha, float P, const double* S, hipStream_t st)
{
    if (level < 1 || !d.dense[level] || iters < 1 || iters > 2) throw std::logic_error("geo_dense: the level or the settings do not fit");
    const int n = d.subtree[level].n;
    const double* Sr = S ? S : d.idle;
    auto launch = [&](auto m, auto po) {
        k::geo_dense<decltype(m)::value, decltype(po)::value><<<n, 512, 0, st>>>(view(d), d.dense[level], level, iters, X, T, B,
                                                                                one_over_alpha, P, Sr);
    };
    using G = std::integral_constant<int, k::GEO_GMG>;
    using M = std::integral_constant<int, k::GEO_CMG>;
    if (mode == k::GEO_GMG && post) launch(G{}, std::true_type{});
    else if (mode == k::GEO_GMG) launch(G{}, std::false_type{});
    else if (post) launch(M{}, std::true_type{});
    else launch(M{}, std::false_type{});
}

void launch_geo_root(const DevGrid& d, int mode, int iters, float* X, const float* B, const double* S, hipStream_t st)
{
    if (!d.root_alone || iters < 0) throw std::logic_error("geo_root: level 0 is not a single tile");
    const int t = d.subtree[0].order[0];
    if (mode == k::GEO_GMG) k::geo_root<k::GEO_GMG><<<1, 256, 0, st>>>(view(d), t, iters, X, B, S ? S : d.idle);
    else k::geo_root<k::GEO_CMG><<<1, 256, 0, st>>>(view(d), t, iters, X, B, S ? S : d.idle);
}

void launch_accumulate_ghosts_add(const DevGrid& d, float* Y, float coeff, const double* S, hipStream_t st)
{
    if (d.ghosts.n <= 0) return;
    k::accumulate_add<<<d.ghosts.n, 64, 0, st>>>(view(d), d.ghosts.d, Y, coeff, S);
}

void launch_residual_interior(const DevGrid& d, const float* B, float* AX, hipStream_t st)
{
    if (d.leafs.n <= 0) return;
    k::residual_interior_v<<<geo_vector_grid(d, d.leafs.n), 256, 0, st>>>(view(d), d.leafs.d, d.leafs.n, B, AX);
}

void launch_djacobi_update(const DevGrid& d, float* X, const float* R, const float* D, float omega, hipStream_t st)
{
    if (d.leafs.n <= 0) return;
    k::djacobi_update_v<<<geo_vector_grid(d, d.leafs.n), 256, 0, st>>>(view(d), d.leafs.d, d.leafs.n, X, R, D, omega);
}

}  // namespace cmg
