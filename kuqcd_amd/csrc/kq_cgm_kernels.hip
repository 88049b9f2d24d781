// Kernels of one multishift CG iteration (CGM::Invert, inverter_cgm.cpp:42-78)
// with the recurrence scalars kept in device memory, plus the start-up and
// reliable-update kernels of the mixed-precision solver.
//
// Per iteration:  begin (several systems) -> D (p0 -> tmp) -> D + axmy + <p0,s> ->
//                 beta, r += b0 s, |r|^2 -> alpha, x/p update of every live shift
// Reductions are two-stage and deterministic: each workgroup writes one FP64
// partial sum, and every workgroup that needs the total adds the partials in the same fixed
// order. The scalar recurrences run in a workgroup of their own beside the vector update that
// needs the scalar, instead of in one-workgroup kernels between the vector kernels (3-5 us each,
// plus 1.2 us from one kernel to the next: a third of an iteration at 8^4 and 16^4).
#include "kq_cgm_device.h"

namespace kq {

// ------------------------------------------------------------ reduce helpers
// Sum part[0..n) in a fixed order with one workgroup of 256 threads.
__device__ inline double block_reduce_fixed(const double *part, uint32_t n)
{
    __shared__ double lds[256];
    double acc = 0.0;
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x)
        acc += part[i];
    lds[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            lds[threadIdx.x] += lds[threadIdx.x + w];
        __syncthreads();
    }
    return lds[0];
}

// The same sum in every thread of a workgroup of 256: `lds` holds 4 doubles, used by this call alone.
// Four loads in flight: one at a time a sum of 2048 partials is 8 waits in a row (32^4 r update of the
// mixed solve 26.0 -> 23.3 us; 8 in flight leave 1024 partials to the loop's remainder)
__device__ inline double sum_partials(const double *part, uint32_t n, double *lds)
{
    double acc = 0.0;
#pragma unroll 4
    for (uint32_t i = threadIdx.x; i < n; i += 256)
        acc += part[i];
    acc = wave_sum(acc);
    if ((threadIdx.x & (kWave - 1)) == 0)
        lds[threadIdx.x / kWave] = acc;
    __syncthreads();
    return (lds[0] + lds[1]) + (lds[2] + lds[3]);
}

// ------------------------------------------------------------ begin
// One wave: the compact list of the live systems, in system order
template <typename S>
__global__ void __launch_bounds__(64) k_cgm_begin(CgmState<S> *st, int nsys, int *rlist, int *nact, int *any)
{
    const int lane = threadIdx.x;
    int n = 0;
    for (int r0 = 0; r0 < nsys; r0 += 64) {
        const int r = r0 + lane;
        const bool live = r < nsys && st[r].stop == 0 && st[r].pause == 0;
        const unsigned long long m = __ballot(live);
        if (live)
            rlist[n + __popcll(m & ((1ull << lane) - 1ull))] = r;
        n += __popcll(m);
    }
    if (lane == 0) {
        *nact = n;
        *any = n > 0;
    }
}

template <typename S> void cgm_begin(CgmState<S> *st, const CgmLaunch &L, hipStream_t stream)
{
    hipLaunchKernelGGL(k_cgm_begin<S>, dim3(1), dim3(64), 0, stream, st, L.nsys, L.rlist, L.nact, L.any);
    KQ_HIP_CHECK(hipGetLastError());
}

// System of list slot `slot`, or -1 when the slot is empty. Without a list (a runner of one
// system) the flag says whether the system iterates: `live` for the hopping terms and the r update,
// its copy `run` for the x/p update, whose scalar workgroup rewrites `live`.
__device__ inline int system_of(int slot, const int *rlist, const int *nact, const int *flag)
{
    if (nact == nullptr)
        return *flag != 0 ? 0 : -1;
    return slot < *nact ? rlist[slot] : -1;
}

// ------------------------------------------------------------ partial sums of large lattices
// out[r][b] = sum of slice b of the kFoldParts slices of part[r][0..n)
template <typename S>
__global__ void __launch_bounds__(256) k_fold_partials(const CgmState<S> *st, const int *rlist, const int *nact,
                                                       const double *part, uint32_t n, double *out)
{
    __shared__ double lds[4];
    const int r = system_of(blockIdx.y, rlist, nact, &st[0].live);
    if (r < 0)
        return;
    const uint32_t per = (n + kFoldParts - 1) / kFoldParts, i0 = blockIdx.x * per;
    const uint32_t m = i0 >= n ? 0u : min(per, n - i0);
    const double v = sum_partials(part + (size_t)r * n + i0, m, lds);
    if (threadIdx.x == 0)
        out[(size_t)r * kFoldParts + blockIdx.x] = v;
}

// ------------------------------------------------------------ beta, r += b0 s, |r|^2
// beta_0 = -|r|^2 / <p0, s>, then r += beta_0 s with the partial sums of |r|^2
// (inverter_cgm.cpp:47-58). The last workgroup of each system runs the zeta/beta recurrences of its
// shifted systems instead, one shift per thread; no other workgroup reads what it writes. The FP
// contraction is switched off so the recurrence rounds exactly as written; the double literal 1.0
// of the reference keeps its type (the denominator is formed in double for S=float).
// HBM-bound at 32^4 (r, s in, r and the history slot out: 101 MB in 20 us, FP64); the sum of the partials
// costs every workgroup about 1 us of L2 reads (16 KB at 32^4), hence at most kBlasMaxBlocks of
// them, each with several site ranges.
template <typename S, typename VR>
__global__ void __launch_bounds__(kBlasNT) k_cgm_update_r(CgmState<S> *st, Vec<VR> r, Vec<VR> s, const int *rlist,
                                                          const int *nact, const double *part_a, uint32_t na,
                                                          double *part_b, c2_t<VR> *rhist, double *shist)
{
#pragma clang fp contract(off)
    using V2 = c2_t<VR>;
    static_assert(kBlasNT == 256, "sum_partials");
    __shared__ double lsum[4], lds[kBlasNT / kWave];
    const int rh = system_of(blockIdx.y, rlist, nact, &st[0].live);
    const uint32_t nb = gridDim.x - 1;  // workgroups over the sites; the last one has the scalars
    const bool scalars = blockIdx.x == nb;
    if (rh < 0) {
        if (nact == nullptr && scalars && threadIdx.x == 0)
            st[0].run = 0;
        return;
    }
    // the first site range is requested before the partials are summed
    V2 rv[3], sv[3];
    uint32_t i = blockIdx.x * kBlasNT + threadIdx.x;
    if (!scalars && i < r.Vh) {
        r.load(rh, i, rv);
        s.load(rh, i, sv);
    }
    const double pAp = sum_partials(part_a + (size_t)rh * na, na, lsum);
    CgmState<S> &c = st[rh];
    const S B0 = -c.rr / (S)pAp;
    if (scalars) {
        // every thread reads the values the shifted updates share before any thread writes
        const S Bm1 = c.Bm1, a0 = c.a[0];
        const int mt = c.maxTerm;
        const bool rec = shist != nullptr && c.dslot >= 0 && c.hist < kHistMax;
        double *h = rec ? shist + hist_scalar_index(c.dslot, c.hist, 0, 0) : nullptr;
        __syncthreads();
        // one shifted system per thread; each touches only its own entries
        for (int j = 1 + (int)threadIdx.x; j < mt; j += blockDim.x) {
            const S zm1 = c.Zm1[j], z = c.Z[j];
            const S num = Bm1 * zm1;
            const S t1 = B0 * a0 * (zm1 - z);
            const S t2 = zm1 * Bm1;
            const S t3 = c.shift[j] * B0;
            const S rr1 = (S)((double)num / ((double)t1 + (double)t2 * (1.0 - (double)t3)));
            const S znew = z * rr1, bnew = B0 * rr1;
            c.Zm1[j] = z;
            c.Z[j] = znew;
            c.B[j] = bnew;
            if (rec) {
                h[j] = (double)bnew;
                h[kMaxShift + j] = (double)znew;
            }
        }
        if (threadIdx.x == 0) {
            c.B[0] = B0;
            c.Bm1 = B0;
            c.rr_prev = c.rr;
            c.maxTermPrev = mt;
            c.run = 1;
            if (rec) {
                h[0] = (double)B0;
                h[kMaxShift] = (double)c.Z[0];
            }
        }
        return;
    }
    const VR b0 = (VR)B0;
    const int ds = c.dslot, hj = c.hist;
    V2 *hist = (rhist != nullptr && ds >= 0 && hj < kHistMax) ? rhist + ((size_t)ds * kHistMax + hj) * 3 * r.Vh : nullptr;
    double acc = 0.0;
    while (i < r.Vh) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            rv[k].x = fmadd(b0, sv[k].x, rv[k].x);
            rv[k].y = fmadd(b0, sv[k].y, rv[k].y);
            acc += (double)rv[k].x * (double)rv[k].x + (double)rv[k].y * (double)rv[k].y;
        }
        r.store(rh, i, rv);
        if (hist != nullptr) {
#pragma unroll
            for (int k = 0; k < 3; ++k)
                st_nt(hist + (size_t)k * r.Vh + i, rv[k]);
        }
        i += nb * kBlasNT;
        if (i < r.Vh) {
            r.load(rh, i, rv);
            s.load(rh, i, sv);
        }
    }
    const double tot = block_sum<kBlasNT>(acc, lds);
    if (threadIdx.x == 0)
        part_b[(size_t)rh * nb + blockIdx.x] = tot;
}

template <typename S, typename VR>
void cgm_update_r(CgmState<S> *st, Vec<VR> r, Vec<VR> s, const CgmLaunch &L, hipStream_t stream)
{
    const double *part = L.part_a;
    uint32_t na = L.nblk_dsl;
    if (na > kFoldAbove) {
        hipLaunchKernelGGL(k_fold_partials<S>, dim3(kFoldParts, L.nlaunch), dim3(256), 0, stream, st, L.rlist, L.nact,
                           L.part_a, na, L.part_f);
        KQ_HIP_CHECK(hipGetLastError());
        part = L.part_f;
        na = kFoldParts;
    }
    hipLaunchKernelGGL((k_cgm_update_r<S, VR>), dim3(cgm_update_nblk(L.Vh) + 1, L.nlaunch), dim3(kBlasNT), 0, stream, st,
                       r, s, L.rlist, L.nact, part, na, L.part_b, static_cast<c2_t<VR> *>(L.rhist), L.shist);
    KQ_HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------------------ alpha, x/p update
// |r|^2, alpha_0 = |r_new|^2 / |r_old|^2, then x_k -= beta_k p_k and p_k = zeta_k r + alpha_k p_k
// (inverter_cgm.cpp:58-69). The last workgroup of each system instead records the alphas, drops
// converged shifts from the end, counts the iteration and sets the stop and pause flags
// (inverter_cgm.cpp:70-78); the others read none of the fields it writes (rr_prev, maxTermPrev, run
// and the betas and zetas were written by k_cgm_update_r).
template <typename S, typename VR, typename XR>
__global__ void __launch_bounds__(kBlasNT) k_cgm_update_p(CgmState<S> *st, XR *x, VR *p, Vec<VR> r, const size_t *off,
                                                          const int *rlist, const int *nact, const double *part_b,
                                                          double *shist)
{
#pragma clang fp contract(off)
    using V2 = c2_t<VR>;
    using X2 = c2_t<XR>;
    __shared__ double lsum[4];
    const int rh = system_of(blockIdx.y, rlist, nact, &st[0].run);
    if (rh < 0)
        return;
    const uint32_t nb = gridDim.x - 1, Vh = r.Vh;
    // the first site range of r and p_0 is requested before the partials are summed
    V2 *p0 = reinterpret_cast<V2 *>(p) + off[rh];
    V2 rv[3], pv[3];
    uint32_t i = blockIdx.x * kBlasNT + threadIdx.x;
    const auto fetch = [&] {
        r.load(rh, i, rv);
#pragma unroll
        for (int k = 0; k < 3; ++k)
            pv[k] = ld_nt(p0 + (size_t)k * Vh + i);
    };
    if (blockIdx.x < nb && i < Vh)
        fetch();
    const double l2_d = sum_partials(part_b + (size_t)rh * nb, nb, lsum);
    CgmState<S> &c = st[rh];
    const S lambda2 = (S)l2_d;
    const S a0 = lambda2 / c.rr_prev;
    const S B0 = c.B[0];
    const int mt = c.maxTermPrev;
    const bool defer = c.dslot >= 0;
    if (blockIdx.x == nb) {
        cgm_finish_iteration(c, l2_d, shist);
        return;
    }
    // a system with deferred solution updates keeps only p_0 current (its x_k and p_k, k >= 1,
    // are brought up to date by the next segment fold)
    const int m = defer ? 1 : mt;
    X2 *x0 = reinterpret_cast<X2 *>(x) + off[rh];
    while (i < Vh) {
        for (int k = 0; k < m; ++k) {
            const size_t base = (size_t)k * 3 * Vh + i;
            const S bk = c.B[k], zk = c.Z[k];
            const VR z = (VR)zk, a = (VR)(k == 0 ? a0 : a0 * zk * bk / (c.Zm1[k] * B0));
            const XR b = (XR)bk;
            V2 *pp = p0 + base;
            X2 *xx = x0 + base;
            if (k > 0) {
#pragma unroll
                for (int cc = 0; cc < 3; ++cc)
                    pv[cc] = ld_nt(pp + (size_t)cc * Vh);
            }
            // streaming accesses except the store of the unshifted direction p_0,
            // which the next hopping term gathers: the solutions and the shifted
            // directions are not touched again before the next update
#pragma unroll
            for (int cc = 0; cc < 3; ++cc) {
                if (!defer) {
                    X2 xv = ld_nt(xx + (size_t)cc * Vh);
                    xv.x = fmadd(-b, (XR)pv[cc].x, xv.x);
                    xv.y = fmadd(-b, (XR)pv[cc].y, xv.y);
                    st_nt(xx + (size_t)cc * Vh, xv);
                }
                V2 np;
                np.x = fmadd(z, rv[cc].x, a * pv[cc].x);
                np.y = fmadd(z, rv[cc].y, a * pv[cc].y);
                if (k == 0)
                    pp[(size_t)cc * Vh] = np;
                else
                    st_nt(pp + (size_t)cc * Vh, np);
            }
        }
        i += nb * kBlasNT;
        if (i < Vh)
            fetch();
    }
}

template <typename S, typename VR, typename XR>
void cgm_update_p(CgmState<S> *st, XR *x, VR *p, Vec<VR> r, const CgmLaunch &L, hipStream_t stream)
{
    hipLaunchKernelGGL((k_cgm_update_p<S, VR, XR>), dim3(cgm_update_nblk(L.Vh) + 1, L.nlaunch), dim3(kBlasNT), 0, stream,
                       st, x, p, r, L.off, L.rlist, L.nact, L.part_b, L.shist);
    KQ_HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------------------ start of systems
template <typename S>
__global__ void __launch_bounds__(256) k_cgm_init_list(CgmState<S> *st, const int *list, const int *n,
                                                       const double *part, uint32_t nblk)
{
    const int slot = blockIdx.x;
    if (*n <= slot)
        return;
    const int r = list[slot];
    const double rr = block_reduce_fixed(part + (size_t)r * nblk, nblk);
    if (threadIdx.x != 0)
        return;
    CgmState<S> &c = st[r];
    c.rr = (S)rr;
    c.Bm1 = (S)1.0;
    for (int k = 0; k < kMaxShift; ++k) {
        c.a[k] = (S)0.0;
        c.B[k] = (S)1.0;
        c.Z[k] = (S)1.0;
        c.Zm1[k] = (S)1.0;
    }
    c.maxTerm = c.nshift;
    c.maxTermUpd = c.nshift;
    c.maxTermFold = c.nshift;
    c.r2max = rr;
    c.iter = 0;
    c.pause = 0;
    c.discard = 0;
    c.hist = 0;
    // the reference's do-while runs at least one iteration even for max_iter <= 0
    c.stop = (c.nshift <= 0) ? 1 : 0;
    c.run = 0;
    c.live = !c.stop;
}

template <typename S>
void cgm_init_list(CgmState<S> *st, const int *list, const int *n, int nsys, const double *part, uint32_t nblk,
                   hipStream_t stream)
{
    hipLaunchKernelGGL(k_cgm_init_list<S>, dim3(nsys), dim3(256), 0, stream, st, list, n, part, nblk);
    KQ_HIP_CHECK(hipGetLastError());
}

template <typename S, typename VR>
__global__ void __launch_bounds__(kBlasNT) k_copy_r_to_p(const CgmState<S> *st, Vec<VR> r, VR *p, const size_t *off,
                                                         const int *list, const int *n)
{
    using V2 = c2_t<VR>;
    const int slot = blockIdx.y;
    if (*n <= slot)
        return;
    const int rh = list[slot];
    const uint32_t i = blockIdx.x * kBlasNT + threadIdx.x;
    const uint32_t Vh = r.Vh;
    if (i >= Vh)
        return;
    V2 rv[3];
    r.load(rh, i, rv);
    const int m = st[rh].nshift;
    for (int k = 0; k < m; ++k) {
        V2 *pp = reinterpret_cast<V2 *>(p) + off[rh] + (size_t)k * 3 * Vh + i;
#pragma unroll
        for (int c = 0; c < 3; ++c)
            pp[(size_t)c * Vh] = rv[c];
    }
}

template <typename S, typename VR>
void copy_r_to_p(const CgmState<S> *st, Vec<VR> r, VR *p, const size_t *off, const int *list, const int *n, int nsys,
                 hipStream_t stream)
{
    hipLaunchKernelGGL((k_copy_r_to_p<S, VR>), dim3(blas_nblk(r.Vh), nsys), dim3(kBlasNT), 0, stream, st, r, p, off,
                       list, n);
    KQ_HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------------------ reliable updates
template <typename VR>
__global__ void __launch_bounds__(kBlasNT) k_rel_residual(const double *b, const double *ax, Vec<VR> r_lo,
                                                          const int *list, const int *n, double *part, uint32_t nblk)
{
    using V2 = c2_t<VR>;
    __shared__ double lds[kBlasNT / kWave];
    const int slot = blockIdx.y;
    if (*n <= slot)
        return;
    const int rh = list[slot];
    const uint32_t Vh = r_lo.Vh;
    const uint32_t i = blockIdx.x * kBlasNT + threadIdx.x;
    double acc = 0.0;
    if (i < Vh) {
        V2 o[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const size_t e = ((size_t)rh * 3 + c) * Vh + i;
            const double2 bb = reinterpret_cast<const double2 *>(b)[e];
            const double2 aa = reinterpret_cast<const double2 *>(ax)[e];
            const double rx = bb.x - aa.x, ry = bb.y - aa.y;
            acc += rx * rx + ry * ry;
            o[c].x = (VR)rx;
            o[c].y = (VR)ry;
        }
        r_lo.store(rh, i, o);
    }
    const double tot = block_sum<kBlasNT>(acc, lds);
    if (threadIdx.x == 0)
        part[(size_t)rh * nblk + blockIdx.x] = tot;
}

template <typename VR>
void rel_residual(const double *b, const double *ax, Vec<VR> r_lo, const int *list, const int *n, int nsys,
                  double *part, uint32_t nblk, hipStream_t stream)
{
    hipLaunchKernelGGL(k_rel_residual<VR>, dim3(nblk, nsys), dim3(kBlasNT), 0, stream, b, ax, r_lo, list, n, part,
                       nblk);
    KQ_HIP_CHECK(hipGetLastError());
}

template <typename S>
__global__ void __launch_bounds__(256) k_rel_set_rr(CgmState<S> *st, const int *list, const int *n,
                                                    const double *part, uint32_t nblk)
{
    const int slot = blockIdx.x;
    if (*n <= slot)
        return;
    const int rh = list[slot];
    const double rr = block_reduce_fixed(part + (size_t)rh * nblk, nblk);
    if (threadIdx.x == 0) {
        st[rh].rr = (S)rr;
        st[rh].r2max = rr;
        st[rh].discard = 0;
    }
}

template <typename S>
void rel_set_rr(CgmState<S> *st, const int *list, const int *n, int nsys, const double *part, uint32_t nblk,
                hipStream_t stream)
{
    hipLaunchKernelGGL(k_rel_set_rr<S>, dim3(nsys), dim3(256), 0, stream, st, list, n, part, nblk);
    KQ_HIP_CHECK(hipGetLastError());
}

template <typename S> __global__ void k_cgm_restart_list(CgmState<S> *st, const int *list, const int *n)
{
    const int slot = blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= *n)
        return;
    CgmState<S> &c = st[list[slot]];
    c.Bm1 = (S)1.0;
    for (int k = 0; k < kMaxShift; ++k) {
        c.a[k] = (S)0.0;
        c.B[k] = (S)1.0;
        c.Z[k] = (S)1.0;
        c.Zm1[k] = (S)1.0;
    }
    c.r2max = (double)c.rr;
    c.pause = 0;
    c.live = !c.stop;
    c.hist = 0;
}

template <typename S> void cgm_restart_list(CgmState<S> *st, const int *list, const int *n, int nsys, hipStream_t stream)
{
    hipLaunchKernelGGL(k_cgm_restart_list<S>, dim3((nsys + 63) / 64), dim3(64), 0, stream, st, list, n);
    KQ_HIP_CHECK(hipGetLastError());
}

template <typename S, typename VR>
__global__ void __launch_bounds__(kBlasNT) k_rel_fold(const CgmState<S> *st, double *x_hi, VR *x_lo,
                                                      const size_t *off, uint32_t Vh, const int *list, const int *n)
{
    using V2 = c2_t<VR>;
    const int slot = blockIdx.y;
    if (*n <= slot)
        return;
    const int rh = list[slot];
    const size_t n3 = (size_t)3 * Vh;
    const size_t i = (size_t)blockIdx.x * kBlasNT + threadIdx.x;
    if (i >= n3)
        return;
    const int m = st[rh].maxTermFold;
    const int discard = st[rh].discard, live = st[rh].maxTerm;
    // streaming accesses except the store of the unshifted solution, which the FP64
    // hopping term of the reliable update reads next
    for (int k = 0; k < m; ++k) {
        const size_t e = off[rh] + (size_t)k * n3 + i;
        V2 *xl = reinterpret_cast<V2 *>(x_lo) + e;
        double2 *xh = reinterpret_cast<double2 *>(x_hi) + e;
        if (fold_keeps(discard, k, live)) {
            const V2 l = ld_nt(xl);
            double2 h = ld_nt(xh);
            h.x += (double)l.x;
            h.y += (double)l.y;
            if (k == 0)
                *xh = h;
            else
                st_nt(xh, h);
        }
        V2 z;
        z.x = 0;
        z.y = 0;
        st_nt(xl, z);
    }
}

template <typename S, typename VR>
void rel_fold(CgmState<S> *st, double *x_hi, VR *x_lo, const size_t *off, uint32_t Vh, const int *list, const int *n,
              int nsys, hipStream_t stream)
{
    const size_t n3 = (size_t)3 * Vh;
    hipLaunchKernelGGL((k_rel_fold<S, VR>), dim3((unsigned)((n3 + kBlasNT - 1) / kBlasNT), nsys), dim3(kBlasNT), 0,
                       stream, st, x_hi, x_lo, off, Vh, list, n);
    KQ_HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------------------ deferred solution updates
// One workgroup per listed system, one thread per (shift k < maxTermFold, term m): the start
// vector (m = -1) or recorded residual m; each forms its pair of coefficients in O(J).
template <typename S>
__global__ void __launch_bounds__(256) k_seg_coef(const CgmState<S> *st, const double *shist, double *coef,
                                                  const int *list, const int *n)
{
    const int slot = blockIdx.x;
    if (*n <= slot)
        return;
    const CgmState<S> &c = st[list[slot]];
    if (c.dslot < 0)
        return;
    const double *h = shist + hist_scalar_index(c.dslot, 0, 0, 0);
    const int terms = kHistMax + 1;
    for (int idx = threadIdx.x; idx < c.maxTermFold * terms; idx += blockDim.x) {
        const int k = idx / terms, m = idx % terms - 1;
        double cx, cp;
        seg_coefficient(h, c.hist, k, m, fold_keeps(c.discard, k, c.maxTerm), cx, cp);
        double *o = coef + ((size_t)c.dslot * kMaxShift + k) * kCoefStride;
        o[1 + m] = cx;                // m = -1: o[0]
        o[kHistMax + 2 + m] = cp;     // m = -1: o[kHistMax + 1]
    }
}

template <typename S>
void seg_coef(const CgmState<S> *st, const double *shist, double *coef, const int *list, const int *n, int nsys,
              hipStream_t stream)
{
    hipLaunchKernelGGL(k_seg_coef<S>, dim3(nsys), dim3(256), 0, stream, st, shist, coef, list, n);
    KQ_HIP_CHECK(hipGetLastError());
}

// One thread per complex entry of a vector. Workgroups are dealt to the 8 XCDs round robin
// (linear id % 8), so blockIdx.x = 8 (k + kmax * (y / 8)) + y % 8 for shift k and site range y:
// the kmax workgroups of one site range run back to back on one XCD and read its recorded
// residuals once into that XCD's L2.
template <typename S, typename VR, typename XR>
__global__ void __launch_bounds__(kBlasNT) k_seg_fold(const CgmState<S> *st, const double *coef, XR *x, VR *p,
                                                      const VR *p0snap, const VR *rhist, const size_t *off,
                                                      uint32_t Vh, const int *list, const int *n, int kmax)
{
    using V2 = c2_t<VR>;
    using X2 = c2_t<XR>;
    const int slot = blockIdx.z;
    const uint32_t rest = blockIdx.x / 8;
    const int k = (int)(rest % (uint32_t)kmax);
    const size_t y = (size_t)(rest / (uint32_t)kmax) * 8 + blockIdx.x % 8;
    if (*n <= slot)
        return;
    const int rh = list[slot];
    const CgmState<S> &c = st[rh];
    if (c.dslot < 0 || k >= c.maxTermFold)
        return;
    const size_t n3 = (size_t)3 * Vh;
    const size_t e = y * kBlasNT + threadIdx.x;
    if (e >= n3)
        return;
    const bool keep_x = fold_keeps(c.discard, k, c.maxTerm);
    const bool upd_p = k >= 1 && k < c.maxTerm;
    if (!keep_x && !upd_p)
        return;
    const int J = c.hist < kHistMax ? c.hist : kHistMax;
    const double *cf = coef + ((size_t)c.dslot * kMaxShift + k) * kCoefStride;
    const size_t pe = off[rh] + (size_t)k * n3 + e;
    const V2 ps = (k == 0) ? reinterpret_cast<const V2 *>(p0snap)[(size_t)c.dslot * n3 + e]
                           : ld_nt(reinterpret_cast<const V2 *>(p) + pe);
    double xr = cf[0] * (double)ps.x, xi = cf[0] * (double)ps.y;
    double pr = cf[kHistMax + 1] * (double)ps.x, pi = cf[kHistMax + 1] * (double)ps.y;
    const V2 *rh_base = reinterpret_cast<const V2 *>(rhist) + (size_t)c.dslot * kHistMax * n3 + e;
    for (int j = 0; j < J; ++j) {
        const V2 rv = rh_base[(size_t)j * n3];
        xr += cf[1 + j] * (double)rv.x;
        xi += cf[1 + j] * (double)rv.y;
        pr += cf[kHistMax + 2 + j] * (double)rv.x;
        pi += cf[kHistMax + 2 + j] * (double)rv.y;
    }
    if (keep_x) {
        X2 *xh = reinterpret_cast<X2 *>(x) + pe;
        X2 h = ld_nt(xh);
        h.x = (XR)((double)h.x + xr);
        h.y = (XR)((double)h.y + xi);
        // the unshifted solution is read next by the FP64 hopping term of a reliable update
        if (k == 0)
            *xh = h;
        else
            st_nt(xh, h);
    }
    if (upd_p) {
        V2 np;
        np.x = (VR)pr;
        np.y = (VR)pi;
        st_nt(reinterpret_cast<V2 *>(p) + pe, np);
    }
}

template <typename S, typename VR, typename XR>
void seg_fold(const CgmState<S> *st, const double *coef, XR *x, VR *p, const VR *p0snap, const VR *rhist,
              const size_t *off, uint32_t Vh, const int *list, const int *n, int nsys, int kmax, hipStream_t stream)
{
    if (kmax <= 0)
        return;
    const size_t n3 = (size_t)3 * Vh;
    const size_t nb8 = (n3 + 8 * kBlasNT - 1) / (8 * kBlasNT);  // site ranges per XCD
    const size_t gx = 8 * (size_t)kmax * nb8;
    if (kmax > kMaxShift || gx > 0x7fffffffu)
        throw std::invalid_argument("seg_fold: grid too large");
    hipLaunchKernelGGL((k_seg_fold<S, VR, XR>), dim3((unsigned)gx, 1, nsys), dim3(kBlasNT), 0, stream, st, coef, x, p,
                       p0snap, rhist, off, Vh, list, n, kmax);
    KQ_HIP_CHECK(hipGetLastError());
}

// p0snap = p_0 and hist = 0 for the listed systems with a history slot
template <typename S, typename VR>
__global__ void __launch_bounds__(kBlasNT) k_seg_reset(CgmState<S> *st, const VR *p, VR *p0snap, const size_t *off,
                                                       uint32_t Vh, const int *list, const int *n)
{
    using V2 = c2_t<VR>;
    const int slot = blockIdx.y;
    if (*n <= slot)
        return;
    const int rh = list[slot];
    const int ds = st[rh].dslot;
    if (ds < 0)
        return;
    const size_t n3 = (size_t)3 * Vh;
    const size_t e = (size_t)blockIdx.x * kBlasNT + threadIdx.x;
    if (e < n3)
        reinterpret_cast<V2 *>(p0snap)[(size_t)ds * n3 + e] = reinterpret_cast<const V2 *>(p)[off[rh] + e];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        st[rh].hist = 0;
        // with one shift left the system goes back to per-iteration updates of x_0 and p_0 (its
        // x_lo, never written while deferred, is zero): the deferral saves nothing there, and
        // x_0 then follows the FP32 p_0 the operator was applied to, as in CGM::Invert
        if (st[rh].maxTerm <= 1)
            st[rh].dslot = -1;
    }
}

template <typename S, typename VR>
void seg_reset(CgmState<S> *st, const VR *p, VR *p0snap, const size_t *off, uint32_t Vh, const int *list, const int *n,
               int nsys, hipStream_t stream)
{
    const size_t n3 = (size_t)3 * Vh;
    hipLaunchKernelGGL((k_seg_reset<S, VR>), dim3((unsigned)((n3 + kBlasNT - 1) / kBlasNT), nsys), dim3(kBlasNT), 0,
                       stream, st, p, p0snap, off, Vh, list, n);
    KQ_HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------------------ true residuals
__global__ void __launch_bounds__(kBlasNT) k_resid2(const double2 *b, const double2 *ax, const int *list, uint32_t Vh,
                                                    double *part, uint32_t nblk)
{
    __shared__ double lds[kBlasNT / kWave];
    const int k = list ? list[blockIdx.y] : (int)blockIdx.y;
    const uint32_t i = blockIdx.x * kBlasNT + threadIdx.x;
    double acc = 0.0;
    if (i < Vh) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double2 bb = b[(size_t)c * Vh + i];
            const double2 aa = ax[((size_t)k * 3 + c) * Vh + i];
            const double rx = bb.x - aa.x, ry = bb.y - aa.y;
            acc += rx * rx + ry * ry;
        }
    }
    const double tot = block_sum<kBlasNT>(acc, lds);
    if (threadIdx.x == 0)
        part[(size_t)k * nblk + blockIdx.x] = tot;
}

void resid2_partial(const double *b, const double *ax, int nk, const int *list, uint32_t Vh, double *part,
                    uint32_t nblk, hipStream_t stream)
{
    if (nk <= 0)
        return;
    hipLaunchKernelGGL(k_resid2, dim3(nblk, nk), dim3(kBlasNT), 0, stream, reinterpret_cast<const double2 *>(b),
                       reinterpret_cast<const double2 *>(ax), list, Vh, part, nblk);
    KQ_HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------------------ generic dot
template <typename VR>
__global__ void __launch_bounds__(kBlasNT) k_dot_partial(Vec<VR> x, Vec<VR> y, double *part, uint32_t nblk,
                                                         const int *list, const int *n)
{
    using V2 = c2_t<VR>;
    __shared__ double lds[kBlasNT / kWave];
    if (n != nullptr && *n <= (int)blockIdx.y)
        return;
    const int rh = list ? list[blockIdx.y] : (int)blockIdx.y;
    const uint32_t i = blockIdx.x * kBlasNT + threadIdx.x;
    double acc = 0.0;
    if (i < x.Vh) {
        V2 a[3], b[3];
        x.load(rh, i, a);
        y.load(rh, i, b);
#pragma unroll
        for (int c = 0; c < 3; ++c)
            acc += (double)a[c].x * (double)b[c].x + (double)a[c].y * (double)b[c].y;
    }
    const double tot = block_sum<kBlasNT>(acc, lds);
    if (threadIdx.x == 0)
        part[(size_t)rh * nblk + blockIdx.x] = tot;
}

template <typename VR>
void vec_dot_partial(Vec<VR> x, Vec<VR> y, int nrhs, double *part, uint32_t nblk, hipStream_t stream, const int *list,
                     const int *n)
{
    hipLaunchKernelGGL(k_dot_partial<VR>, dim3(nblk, nrhs), dim3(kBlasNT), 0, stream, x, y, part, nblk, list, n);
    KQ_HIP_CHECK(hipGetLastError());
}

__global__ void __launch_bounds__(256) k_reduce_partials(const double *part, uint32_t nblk, double *out)
{
    const int r = blockIdx.x;
    const double v = block_reduce_fixed(part + (size_t)r * nblk, nblk);
    if (threadIdx.x == 0)
        out[r] = v;
}

void reduce_partials(const double *part, uint32_t nblk, int nrhs, double *out, hipStream_t stream)
{
    hipLaunchKernelGGL(k_reduce_partials, dim3(nrhs), dim3(256), 0, stream, part, nblk, out);
    KQ_HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------------------ instantiations
#define KQ_INST_S(S)                                                                                          \
    template void cgm_begin<S>(CgmState<S> *, const CgmLaunch &, hipStream_t);                                \
    template void cgm_init_list<S>(CgmState<S> *, const int *, const int *, int, const double *, uint32_t,    \
                                   hipStream_t);                                                              \
    template void rel_set_rr<S>(CgmState<S> *, const int *, const int *, int, const double *, uint32_t,       \
                                hipStream_t);                                                              \
    template void cgm_restart_list<S>(CgmState<S> *, const int *, const int *, int, hipStream_t);          \
    template void seg_coef<S>(const CgmState<S> *, const double *, double *, const int *, const int *, int,   \
                              hipStream_t);
KQ_INST_S(double)
KQ_INST_S(float)

#define KQ_INST_SV(S, VR)                                                                                      \
    template void cgm_update_r<S, VR>(CgmState<S> *, Vec<VR>, Vec<VR>, const CgmLaunch &, hipStream_t);        \
    template void cgm_update_p<S, VR, VR>(CgmState<S> *, VR *, VR *, Vec<VR>, const CgmLaunch &, hipStream_t); \
    template void rel_fold<S, VR>(CgmState<S> *, double *, VR *, const size_t *, uint32_t, const int *,        \
                                  const int *, int, hipStream_t);                                             \
    template void copy_r_to_p<S, VR>(const CgmState<S> *, Vec<VR>, VR *, const size_t *, const int *,          \
                                     const int *, int, hipStream_t);                                          \
    template void seg_fold<S, VR, double>(const CgmState<S> *, const double *, double *, VR *, const VR *,    \
                                          const VR *, const size_t *, uint32_t, const int *, const int *, int, int, \
                                          hipStream_t);                                                        \
    template void seg_reset<S, VR>(CgmState<S> *, const VR *, VR *, const size_t *, uint32_t, const int *,     \
                                   const int *, int, hipStream_t);
KQ_INST_SV(double, double)
KQ_INST_SV(float, float)
KQ_INST_SV(double, float)
// the float reference method folds into its FP32 solutions
template void seg_fold<float, float, float>(const CgmState<float> *, const double *, float *, float *, const float *,
                                            const float *, const size_t *, uint32_t, const int *, const int *, int, int,
                                            hipStream_t);

template void rel_residual<float>(const double *, const double *, Vec<float>, const int *, const int *, int,
                                  double *, uint32_t, hipStream_t);
template void rel_residual<double>(const double *, const double *, Vec<double>, const int *, const int *, int,
                                   double *, uint32_t, hipStream_t);
template void vec_dot_partial<double>(Vec<double>, Vec<double>, int, double *, uint32_t, hipStream_t, const int *,
                                      const int *);
template void vec_dot_partial<float>(Vec<float>, Vec<float>, int, double *, uint32_t, hipStream_t, const int *,
                                     const int *);

// ------------------------------------------------------------ small copies
__global__ void __launch_bounds__(256) k_copy_words(const unsigned long long *src, unsigned long long *dst, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        dst[i] = src[i];
}

void copy_words(const void *src, void *dst, size_t bytes, hipStream_t stream)
{
    if (bytes % 8 != 0)
        throw std::invalid_argument("copy_words: size must be a multiple of 8 bytes");
    const size_t n = bytes / 8;
    if (n == 0)
        return;
    const unsigned grid = (unsigned)std::min<size_t>((n + 255) / 256, 64);
    hipLaunchKernelGGL(k_copy_words, dim3(grid), dim3(256), 0, stream,
                       static_cast<const unsigned long long *>(src), static_cast<unsigned long long *>(dst), n);
    KQ_HIP_CHECK(hipGetLastError());
}

__global__ void __launch_bounds__(256) k_set_int_list(const int *src, int *list, int *count, int n)
{
    for (int i = threadIdx.x; i < n; i += 256)
        list[i] = src[i];
    if (threadIdx.x == 0)
        *count = n;
}

void set_int_list(const int *src, int *list, int *count, int n, hipStream_t stream)
{
    hipLaunchKernelGGL(k_set_int_list, dim3(1), dim3(256), 0, stream, src, list, count, n);
    KQ_HIP_CHECK(hipGetLastError());
}

}  // namespace kq
