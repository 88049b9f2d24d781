// Solve drivers behind kq_solve_multishift / _ex / _batched.
#pragma once

#include "kq_context.h"
#include "kq_dslash.h"
#include "kuqcd_hip.h"

namespace kq {

// The reference method (CGM::Invert) in the loaded gauge precision.
KuQCDStatus solve_reference(int slot, void **x, void *b, KuQCDInvertParam &p);

// FP64 or mixed-precision multishift CG for nrhs sources with per-shift FP64
// verification and refinement.
KuQCDStatus solve_extended(int slot, int nrhs, void **x, void **b, KuQCDInvertParam &p, const KqSolveOptions &o,
                           KqSolveReport *rep);

// sum_blk part[k][blk] on the host side
std::vector<double> reduce_host(const double *part_dev, uint32_t nblk, int n, hipStream_t st);

// bytes from device memory d to h (pageable host, pinned host or device memory), synchronous with
// respect to the host; pageable destinations go through pinned chunks (kq_xfer.cpp)
void copy_to_host(void *h, const void *d, size_t bytes, hipStream_t st);
// bytes from h (pageable host, pinned host or device memory) to device memory d, likewise
void copy_from_host(void *d, const void *h, size_t bytes, hipStream_t st);

// true for device memory of any GPU (not host or managed memory), and of the current one
bool on_a_device(const void *p);
bool on_this_device(const void *p);
// true where kernels can read or write a caller's array of `bytes` bytes with elements of `elem` bytes
// themselves: aligned, in device memory of the current GPU and inside one allocation. Other arrays
// go through a copy, which reports what it cannot reach.
bool in_place(const void *p, size_t bytes, size_t elem);

// dst = sigma src - D D src on parity `parity`, src and dst in the caller's host layout in device
// memory (not overlapping), tmp a device vector of the other parity: two launches, not waited for
template <class LF, class LL, typename R>
inline void mdaggm_host(LF fat, LL lng, const Geom &g, const R *src, R *dst, c2_t<R> *tmp, int parity, double sigma,
                        hipStream_t st)
{
    const size_t n3 = (size_t)3 * g.Vh;
    const Vec<R> sv{reinterpret_cast<c2_t<R> *>(const_cast<R *>(src)), g.Vh, n3}, tv{tmp, g.Vh, n3};
    DslashArgs<LF, LL, R> a{};
    a.g = g;
    a.fat = fat;
    a.lng = lng;
    a.nrhs = 1;
    a.dst_parity = 1 - parity;
    a.src = sv;
    a.dst = tv;
    launch_dslash_host(a, LAY_HOST_SRC, EPI_STORE, 1, st);
    a.dst_parity = parity;
    a.src = tv;
    a.dst = Vec<R>{reinterpret_cast<c2_t<R> *>(dst), g.Vh, n3};
    a.aux = sv;
    a.sigma0 = sigma;
    launch_dslash_host(a, LAY_HOST_DST, EPI_AXMY, 1, st);
}

// caller vector (reference layout, HR; host or device memory) -> device SoA vector r of v. Device
// arrays are converted where they lie (an upload through a staging copy took 16 us at 16^4, 5 of
// them the copy and 8 the wait); wait = false leaves the wait for the conversion to the caller,
// who waits for the stream before its own return.
template <typename HR, typename VR> inline void upload_vec(const void *h, Vec<VR> v, int r, DevBuf &stage, hipStream_t st, bool wait = true)
{
    const size_t n = (size_t)6 * v.Vh;
    if (in_place(h, sizeof(HR) * n, sizeof(HR))) {
        vec_host_to_soa<HR, VR>(static_cast<const HR *>(h), v, r, st);
        if (wait)
            KQ_HIP_CHECK(hipStreamSynchronize(st));
        return;
    }
    if (stage.bytes() < sizeof(HR) * n)
        stage.alloc(sizeof(HR) * n);
    copy_from_host(stage.as<void>(), h, sizeof(HR) * n, st);
    vec_host_to_soa<HR, VR>(stage.as<HR>(), v, r, st);
    KQ_HIP_CHECK(hipStreamSynchronize(st));
}

template <typename VR, typename HR> inline void download_vec(Vec<VR> v, int r, void *h, DevBuf &stage, hipStream_t st, bool wait = true)
{
    const size_t n = (size_t)6 * v.Vh;
    if (in_place(h, sizeof(HR) * n, sizeof(HR))) {
        vec_soa_to_host<VR, HR>(v, r, static_cast<HR *>(h), st);
        if (wait)
            KQ_HIP_CHECK(hipStreamSynchronize(st));
        return;
    }
    if (stage.bytes() < sizeof(HR) * n)
        stage.alloc(sizeof(HR) * n);
    vec_soa_to_host<VR, HR>(v, r, stage.as<HR>(), st);
    copy_to_host(h, stage.as<void>(), sizeof(HR) * n, st);
}

// autotuned (nr, nt) for the hopping term
std::pair<int, int> tuned_launch(int slot, int mode, int nrhs);
// occupancy cap (waves per SIMD, 0 = none) measured best for (nr, nt) by tuned_launch
int tuned_cap(int slot, int mode, int nr, int nt);

}  // namespace kq
