// Scalar part of the x/p update, shared by the update's own kernel and by the hopping term that
// applies it on the way (k_dslash_split_p).
#pragma once

#include "kq_cgm_kernels.h"

namespace kq {

// Record the alphas of the iteration whose |r|^2 is l2_d, drop converged shifts from the end, count
// the iteration and set the stop and pause flags (inverter_cgm.cpp:58-78); by one workgroup. The FP
// contraction is switched off so the recurrence rounds exactly as written.
template <typename S> __device__ inline void cgm_finish_iteration(CgmState<S> &c, double l2_d, double *shist)
{
#pragma clang fp contract(off)
    const S lambda2 = (S)l2_d;
    const S a0 = lambda2 / c.rr_prev;
    const S B0 = c.B[0];
    const int mt = c.maxTermPrev;
    const int hj = c.hist;
    const bool rec = shist != nullptr && c.dslot >= 0 && hj < kHistMax;
    double *h = rec ? shist + hist_scalar_index(c.dslot, hj, 2, 0) : nullptr;
    __syncthreads();
    for (int j = 1 + (int)threadIdx.x; j < mt; j += blockDim.x) {
        const S aj = a0 * c.Z[j] * c.B[j] / (c.Zm1[j] * B0);
        c.a[j] = aj;
        if (rec)
            h[j] = (double)aj;
    }
    if (threadIdx.x != 0)
        return;
    c.a[0] = a0;
    c.rr = lambda2;
    c.maxTermUpd = mt;
    if (rec) {
        h[0] = (double)a0;
        h[kMaxShift] = (double)mt;
        c.hist = hj + 1;
    }
    // drop converged shifts from the end of the list (inverter_cgm.cpp:71-76)
    int left = mt;
    while (left > 0) {
        const S lambda = c.Z[left - 1] * c.Z[left - 1] * lambda2;
        if (!((double)lambda < c.tolk[left - 1]))
            break;
        left--;
    }
    c.maxTerm = left;
    const int iter = c.iter + 1;
    c.iter = iter;
    const bool stop = left <= 0 || iter >= c.maxIter;
    const bool pause = c.pause2 > 0.0 && l2_d < c.pause2 * c.r2max;
    if (stop)
        c.stop = 1;
    if (pause)
        c.pause = 1;
    c.live = !stop && !pause;
}

}  // namespace kq
