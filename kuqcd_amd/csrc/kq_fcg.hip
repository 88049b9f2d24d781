// Kernels of the flexible CG: fused vector updates with block partial sums. A vector update that
// needs a scalar adds the partials of the kernel before it itself, in every workgroup and in the same
// fixed order (one-workgroup kernels for beta and alpha took 4.3 and 7.6 us of an iteration at
// 24^4); the check of the residual is a workgroup of its own, since it stops the kernels after it.
#include "kq_fcg.h"

#include <algorithm>

namespace kq {

namespace {

constexpr int kNT = 256;

__device__ __forceinline__ bool halted(const FcgState *st) { return st->stop != 0; }

// block sum of (a, b) into part[2*blk], part[2*blk+1] (b ignored when part2 is false)
template <bool TWO>
__device__ __forceinline__ void block_partial(double a, double b, double *part)
{
    __shared__ double la[kNT / kWave], lb[kNT / kWave];
    a = wave_sum(a);
    if (TWO)
        b = wave_sum(b);
    if ((threadIdx.x & (kWave - 1)) == 0) {
        la[threadIdx.x / kWave] = a;
        if (TWO)
            lb[threadIdx.x / kWave] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double sa = 0.0, sb = 0.0;
        for (int w = 0; w < kNT / kWave; ++w) {
            sa += la[w];
            if (TWO)
                sb += lb[w];
        }
        if (TWO) {
            part[2 * blockIdx.x] = sa;
            part[2 * blockIdx.x + 1] = sb;
        } else {
            part[blockIdx.x] = sa;
        }
    }
}

// sums over k < nblk of the W values part[W*k .. W*k + W), the same in every thread of the workgroup;
// lds: 4*W doubles used by this call alone
template <int W> __device__ __forceinline__ void sum_partials(const double *part, uint32_t nblk, double *lds, double *out)
{
    double s[W];
#pragma unroll
    for (int w = 0; w < W; ++w)
        s[w] = 0.0;
#pragma unroll 4
    for (uint32_t k = threadIdx.x; k < nblk; k += kNT)
#pragma unroll
        for (int w = 0; w < W; ++w)
            s[w] += part[(size_t)W * k + w];
#pragma unroll
    for (int w = 0; w < W; ++w) {
        s[w] = wave_sum(s[w]);
        if ((threadIdx.x & (kWave - 1)) == 0)
            lds[W * (threadIdx.x / kWave) + w] = s[w];
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < W; ++w)
        out[w] = (lds[w] + lds[W + w]) + (lds[2 * W + w] + lds[3 * W + w]);
}

// out[W*b + w] = sum of slice b of the kFoldParts slices of part (large lattices)
constexpr uint32_t kFoldParts = 64;
template <int W>
__global__ void __launch_bounds__(kNT) k_fcg_fold_partials(const FcgState *st, const double *part, uint32_t n,
                                                           double *out)
{
    __shared__ double lds[4 * W];
    if (halted(st))
        return;
    const uint32_t per = (n + kFoldParts - 1) / kFoldParts, i0 = blockIdx.x * per;
    double t[W];
    sum_partials<W>(part + (size_t)W * i0, i0 >= n ? 0u : min(per, n - i0), lds, t);
    if (threadIdx.x == 0)
#pragma unroll
        for (int w = 0; w < W; ++w)
            out[W * blockIdx.x + w] = t[w];
}

__global__ void __launch_bounds__(kNT) k_fcg_dot(const FcgState *st, const float2 *q, const float2 *z, size_t n,
                                                 double *part)
{
    if (halted(st))
        return;
    double re = 0.0, im = 0.0;
    for (size_t i = (size_t)blockIdx.x * kNT + threadIdx.x; i < n; i += (size_t)gridDim.x * kNT) {
        const float2 a = q[i], b = z[i];
        re += (double)a.x * b.x + (double)a.y * b.y;
        im += (double)a.x * b.y - (double)a.y * b.x;
    }
    block_partial<true>(re, im, part);
}

// beta = <q, z> / <p, q> of the previous iteration (0 on a first one), p = z - beta p, partials of <p, r>
__global__ void __launch_bounds__(kNT) k_fcg_p_update(const FcgState *st, const double *part_qz, uint32_t nblk,
                                                      const float2 *z, float2 *p, const float2 *r, size_t n,
                                                      double *part)
{
    __shared__ double lds[8];
    if (halted(st))
        return;
    size_t i = (size_t)blockIdx.x * kNT + threadIdx.x;
    float2 zi = {}, ri = {}, po = {};
    // the vectors' loads run while the partials are summed (p is read on a first iteration as well)
    auto fetch = [&] {
        if (i < n) {
            zi = z[i];
            ri = r[i];
            po = p[i];
        }
    };
    fetch();
    double qz[2];
    sum_partials<2>(part_qz, nblk, lds, qz);
    const bool first = st->first != 0;
    const double pq = st->pq_prev;
    const bool none = first || pq == 0.0;
    const float br = none ? 0.f : (float)(qz[0] / pq), bi = none ? 0.f : (float)(qz[1] / pq);
    double re = 0.0, im = 0.0;
    for (; i < n; i += (size_t)gridDim.x * kNT, fetch()) {
        float2 pi = zi;
        if (!first) {
            pi.x -= br * po.x - bi * po.y;
            pi.y -= br * po.y + bi * po.x;
        }
        p[i] = pi;
        re += (double)pi.x * ri.x + (double)pi.y * ri.y;
        im += (double)pi.x * ri.y - (double)pi.y * ri.x;
    }
    block_partial<true>(re, im, part);
}

// alpha = <p, r> / <p, q>, x += alpha p, r -= alpha q, partials of |r|^2. The last workgroup keeps
// <p, q> for the next beta instead (no other workgroup reads what it writes).
__global__ void __launch_bounds__(kNT) k_fcg_xr_update(FcgState *st, const double *part_pq, uint32_t nblk_pq,
                                                       const double *part_pr, uint32_t nblk_pr, float2 *x, float2 *r,
                                                       const float2 *p, const float2 *q, size_t n, double *part)
{
    __shared__ double lpq[4], lpr[8];
    if (halted(st))
        return;
    const uint32_t nb = gridDim.x - 1;
    size_t i = (size_t)blockIdx.x * kNT + threadIdx.x;
    float2 pi = {}, qi = {}, xi = {}, ri = {};
    auto fetch = [&] {
        if (i < n) {
            pi = p[i];
            qi = q[i];
            xi = x[i];
            ri = r[i];
        }
    };
    if (blockIdx.x < nb)
        fetch();
    double pq, pr[2];
    sum_partials<1>(part_pq, nblk_pq, lpq, &pq);
    if (blockIdx.x == nb) {
        if (threadIdx.x == 0) {
            st->pq_prev = pq;
            st->first = 0;
        }
        return;
    }
    sum_partials<2>(part_pr, nblk_pr, lpr, pr);
    const bool ok = pq > 0.0;
    const float ar = ok ? (float)(pr[0] / pq) : 0.f, ai = ok ? (float)(pr[1] / pq) : 0.f;
    double rr = 0.0;
    for (; i < n; i += (size_t)nb * kNT, fetch()) {
        xi.x += ar * pi.x - ai * pi.y;
        xi.y += ar * pi.y + ai * pi.x;
        ri.x -= ar * qi.x - ai * qi.y;
        ri.y -= ar * qi.y + ai * qi.x;
        x[i] = xi;
        r[i] = ri;
        rr += (double)ri.x * ri.x + (double)ri.y * ri.y;
    }
    block_partial<false>(rr, 0.0, part);
}

__global__ void __launch_bounds__(kNT) k_fcg_check(FcgState *st, const double *part, uint32_t nblk)
{
    __shared__ double lds[4];
    if (halted(st))
        return;
    double rr;
    sum_partials<1>(part, nblk, lds, &rr);
    if (threadIdx.x == 0) {
        st->rr = rr;
        st->iter += 1;
        int reason = 0;
        if (!(rr > st->rr_stop))  // also stops on NaN
            reason = kFcgStopConverged;
        else if (rr <= st->rr_pause)
            reason = kFcgStopPause;
        else if (st->iter >= st->max_iter)
            reason = kFcgStopMaxIter;
        if (reason) {
            st->reason = reason;
            st->stop = 1;
            st->run = 0;
        }
    }
}

__global__ void k_fcg_fold(double2 *x64, float2 *x32, size_t n)
{
    const size_t i = (size_t)blockIdx.x * kNT + threadIdx.x;
    if (i < n) {
        const float2 a = x32[i];
        double2 b = x64[i];
        b.x += a.x;
        b.y += a.y;
        x64[i] = b;
        x32[i] = mk<float2>(0.f, 0.f);
    }
}

__global__ void __launch_bounds__(kNT) k_fcg_residual(const double2 *b, const double2 *ax, double2 *r64,
                                                      float2 *r32, size_t n, double *part)
{
    double rr = 0.0;
    for (size_t i = (size_t)blockIdx.x * kNT + threadIdx.x; i < n; i += (size_t)gridDim.x * kNT) {
        const double2 bi = b[i], ai = ax[i];
        const double2 ri = mk<double2>(bi.x - ai.x, bi.y - ai.y);
        if (r64)
            r64[i] = ri;
        r32[i] = mk<float2>((float)ri.x, (float)ri.y);
        rr += ri.x * ri.x + ri.y * ri.y;
    }
    block_partial<false>(rr, 0.0, part);
}

__global__ void k_fcg_to_f32(const double2 *a, const double2 *b, double scale, float2 *out, size_t n)
{
    const size_t i = (size_t)blockIdx.x * kNT + threadIdx.x;
    if (i < n) {
        double2 v = a[i];
        if (b) {
            const double2 w = b[i];
            v.x -= w.x;
            v.y -= w.y;
        }
        out[i] = mk<float2>((float)(scale * v.x), (float)(scale * v.y));
    }
}

}  // namespace

static uint32_t full_grid(size_t n) { return (uint32_t)((n + kNT - 1) / kNT); }
uint32_t fcg_nblk(size_t n) { return std::min(full_grid(n), kFcgMaxBlocks); }

#define KQ_FCG_LAUNCH(kernel, grid, ...)                                           \
    do {                                                                           \
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(kNT), 0, s, __VA_ARGS__);      \
        KQ_HIP_CHECK(hipGetLastError());                                           \
    } while (0)

// Above this many partials (64 KB) they are first summed in slices: every workgroup of an update
// reads all that are left
constexpr uint32_t kFoldAbove = 8192;
template <int W>
static const double *folded(const FcgState *st, const double *part, uint32_t &n, double *fold, hipStream_t s)
{
    if ((size_t)W * n <= kFoldAbove)
        return part;
    KQ_FCG_LAUNCH(k_fcg_fold_partials<W>, kFoldParts, st, part, n, fold);
    n = kFoldParts;
    return fold;
}

void fcg_dot(const FcgState *st, const float2 *q, const float2 *z, size_t n, double *part, hipStream_t s)
{
    KQ_FCG_LAUNCH(k_fcg_dot, fcg_nblk(n), st, q, z, n, part);
}
void fcg_p_update(const FcgState *st, const double *part_qz, uint32_t nblk, double *fold, const float2 *z, float2 *p,
                  const float2 *r, size_t n, double *part, hipStream_t s)
{
    part_qz = folded<2>(st, part_qz, nblk, fold, s);
    KQ_FCG_LAUNCH(k_fcg_p_update, fcg_nblk(n), st, part_qz, nblk, z, p, r, n, part);
}
void fcg_xr_update(FcgState *st, const double *part_pq, uint32_t nblk_pq, double *fold, const double *part_pr, float2 *x,
                   float2 *r, const float2 *p, const float2 *q, size_t n, double *part, hipStream_t s)
{
    part_pq = folded<1>(st, part_pq, nblk_pq, fold, s);
    KQ_FCG_LAUNCH(k_fcg_xr_update, fcg_nblk(n) + 1, st, part_pq, nblk_pq, part_pr, fcg_nblk(n), x, r, p, q, n, part);
}
void fcg_check(FcgState *st, const double *part, uint32_t nblk, hipStream_t s)
{
    KQ_FCG_LAUNCH(k_fcg_check, 1, st, part, nblk);
}
void fcg_fold(double2 *x64, float2 *x32, size_t n, hipStream_t s)
{
    if (n)
        KQ_FCG_LAUNCH(k_fcg_fold, full_grid(n), x64, x32, n);
}
void fcg_residual(const double2 *b, const double2 *ax, double2 *r64, float2 *r32, size_t n, double *part,
                  hipStream_t s)
{
    if (n)
        KQ_FCG_LAUNCH(k_fcg_residual, fcg_nblk(n), b, ax, r64, r32, n, part);
}

void fcg_to_f32(const double2 *a, const double2 *b, double scale, float2 *out, size_t n, hipStream_t s)
{
    if (n)
        KQ_FCG_LAUNCH(k_fcg_to_f32, full_grid(n), a, b, scale, out, n);
}

}  // namespace kq
