// cmg_inverse.hip -- the FP64 inverse of the level-0 operator on gfx950.
//
// Blocked Gauss-Jordan elimination in blocks of 32 x 32, without pivoting: for a symmetric
// positive definite matrix every pivot is positive and the elimination is stable.  A pivot
// that is not positive is reported, and the caller then takes the pivoted elimination on the
// host.  One launch does one block column K out of place (A to B), a workgroup a block:
//   P = A[K][K]^-1;  B[K][K] = P;  B[K][j] = P A[K][j];  B[i][K] = -A[i][K] P;
//   B[i][j] = A[i][j] - A[i][K] (P A[K][j])
// Every workgroup inverts the pivot block again in its own LDS, which costs no launch and no
// wait; that chain of 32 dependent steps is what bounds a launch at the usual 512 unknowns
// (16 launches of 256 workgroups, one a CU).  (MI355X, 512 unknowns: 16 x 21.7 us; the first
// solve on a new 256^3 sphere octree takes 5.5 ms instead of 12.8 with the elimination of the
// 512 x 1,024 system on 16 host threads.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdexcept>
#include <string>

#include "cmg_device.hpp"
#include "cmg_kernels.hpp"

#pragma clang fp contract(off)

namespace cmg {
namespace k {

constexpr int IB = 32;

// A: ld x ld, `shift` on the n x n unknowns, the identity on the padding
__global__ __launch_bounds__(256) void inverse_init(double* __restrict__ A, int ld, int n, double shift)
{
    const size_t e = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (e >= size_t(ld) * ld) return;
    const int r = int(e / ld), c = int(e % ld);
    A[e] = r < n && c < n ? shift : r == c ? 1.0 : 0.0;
}

// entries (row, column) = (rc >> 16, rc & 0xffff), each place at most once
__global__ __launch_bounds__(256) void inverse_entries(double* __restrict__ A, int ld, const uint32_t* __restrict__ rc,
                                                       const double* __restrict__ v, int m)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= m) return;
    double& a = A[size_t(rc[e] >> 16) * ld + (rc[e] & 0xffffu)];
    a = a + v[e];
}

// block column K of the elimination; B has rows of ldb and keeps its first nb x nb entries
__global__ __launch_bounds__(256) void inverse_step(const double* __restrict__ A, double* __restrict__ B, int ld, int ldb, int nb,
                                                    int K, double floor, int* __restrict__ bad)
{
    __shared__ double P[IB][IB + 1], L[IB][IB + 1], R[IB][IB + 1];
    const int j = blockIdx.x, i = blockIdx.y, tid = threadIdx.x;
    const int r = tid >> 3, c0 = 4 * (tid & 7);   // four entries of a row a thread
    auto block = [&](int bi, int bj) { return A + (size_t(bi) * IB + r) * ld + size_t(bj) * IB + c0; };
    double own[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        P[r][c0 + e] = block(K, K)[e];
        L[r][c0 + e] = block(i, K)[e];
        R[r][c0 + e] = block(K, j)[e];
        own[e] = block(i, j)[e];
    }
    __syncthreads();
    for (int k = 0; k < IB; ++k) {
        const double p = P[k][k], ip = 1.0 / p, f = P[r][k];
        if (i == K && j == K && tid == 0 && !(p > floor)) *bad = 1;
        double v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int c = c0 + e;
            const double row = P[k][c] * ip;
            v[e] = r == k ? (c == k ? ip : row) : (c == k ? -f * ip : P[r][c] - f * row);
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 4; ++e) P[r][c0 + e] = v[e];
        __syncthreads();
    }
    double o[4];
    if (i == K) {
        // P, or P A[K][j]
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            double s = 0.0;
            for (int k = 0; k < IB; ++k) s = fma(P[r][k], R[k][c0 + e], s);
            o[e] = j == K ? P[r][c0 + e] : s;
        }
    } else {
        // S = A[i][K] P, then -S or A[i][j] - S A[K][j]
        double s[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s[e] = 0.0;
            for (int k = 0; k < IB; ++k) s[e] = fma(L[r][k], P[k][c0 + e], s[e]);
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 4; ++e) L[r][c0 + e] = s[e];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            double v = own[e];
            for (int k = 0; k < IB; ++k) v = fma(-L[r][k], R[k][c0 + e], v);
            o[e] = j == K ? -s[e] : v;
        }
    }
    const int row = i * IB + r, col = j * IB + c0;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (row < nb && col + e < nb) B[size_t(row) * ldb + col + e] = o[e];
}

}  // namespace k

bool device_inverse(int n, double shift, const std::vector<uint32_t>& rc, const std::vector<double>& v, double* inv, hipStream_t st)
{
    auto ok = [](hipError_t e) {
        if (e != hipSuccess) throw std::runtime_error(std::string("level-0 inverse: ") + hipGetErrorString(e));
    };
    if (n <= 0 || n > 4096 || rc.size() != v.size()) throw std::logic_error("level-0 inverse: bad size");
    const int nb = (n + k::IB - 1) / k::IB, ld = nb * k::IB, m = int(rc.size());
    // a nearly singular matrix is left to the caller as well
    double top = 0.0;
    for (int e = 0; e < m; ++e)
        if ((rc[e] >> 16) == (rc[e] & 0xffffu)) top = std::max(top, v[e] + shift);
    const double floor = 1e-10 * top;
    const size_t a = size_t(ld) * ld * sizeof(double), ve = (size_t(m) * sizeof(double) + 255) & ~size_t(255);
    char* block = nullptr;
    const hipError_t got = hipMalloc(reinterpret_cast<void**>(&block), 2 * a + ve + size_t(m) * sizeof(uint32_t) + 256);
    if (got == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        return false;   // the caller's elimination takes no device memory
    }
    ok(got);
    int bad = 0;
    try {
        double* A[2] = {reinterpret_cast<double*>(block), reinterpret_cast<double*>(block + a)};
        double* dv = reinterpret_cast<double*>(block + 2 * a);
        int* dbad = reinterpret_cast<int*>(block + 2 * a + ve);
        uint32_t* drc = reinterpret_cast<uint32_t*>(block + 2 * a + ve + 256);
        ok(hipMemcpyAsync(dv, v.data(), size_t(m) * sizeof(double), hipMemcpyHostToDevice, st));
        ok(hipMemcpyAsync(drc, rc.data(), size_t(m) * sizeof(uint32_t), hipMemcpyHostToDevice, st));
        ok(hipMemcpyAsync(dbad, &bad, sizeof(bad), hipMemcpyHostToDevice, st));
        k::inverse_init<<<unsigned((size_t(ld) * ld + 255) / 256), 256, 0, st>>>(A[0], ld, n, shift);
        if (m) k::inverse_entries<<<(m + 255) / 256, 256, 0, st>>>(A[0], ld, drc, dv, m);
        for (int K = 0; K < nb; ++K) {
            const bool last = K == nb - 1;
            k::inverse_step<<<dim3(nb, nb), 256, 0, st>>>(A[K & 1], last ? inv : A[(K + 1) & 1], ld, last ? n : ld,
                                                          last ? n : ld, K, floor, dbad);
        }
        ok(hipGetLastError());
        ok(hipMemcpyAsync(&bad, dbad, sizeof(bad), hipMemcpyDeviceToHost, st));
        ok(hipStreamSynchronize(st));
    } catch (...) {
        (void)hipStreamSynchronize(st);
        (void)hipFree(block);
        throw;
    }
    (void)hipFree(block);
    return bad == 0;
}

}  // namespace cmg
