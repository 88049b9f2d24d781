// HISQ even-odd hopping term (fat 1-hop + Naik 3-hop) on gfx950.
//
// One thread per output site (and per block of NR right-hand sides): the
// 16 links of the site are each read once from HBM with coalesced
// structure-of-arrays loads and applied to the NR gathered neighbour vectors,
// so a batched launch reads every link once for all of its right-hand sides.
// Periodic boundaries are resolved in-kernel from the site coordinates; no
// neighbour tables are read. Follows DiracHISQ::Dslash/FwdDslash/BwdDslash
// (dirac_hisq.cpp:409-502) with the 1/2 and c3000 factors folded into the
// device links.
//
// Implementation header: kq_dslash_*.hip instantiate launch_dslash for the link
// formats (one translation unit per family, so they compile in parallel).
#pragma once

#include "kq_cgm_device.h"
#include "kq_dslash.h"

#include <algorithm>
#include <type_traits>

namespace kq {

// gather the colour vector at site n of right-hand side j (base pointer src[j]); AOS: the caller's
// host layout (a site's three colours together, kq_fields.h) instead of the library's colour planes
template <bool AOS = false, class V2>
__device__ __forceinline__ void gather(const V2 *src, uint32_t n, uint32_t Vh, V2 v[3])
{
    if constexpr (AOS) {
        ld_site(src + (size_t)3 * n, v);
    } else {
#pragma unroll
        for (int c = 0; c < 3; ++c)
            v[c] = src[(size_t)c * Vh + n];
    }
}

// A search direction that is formed where it is gathered: z r + a p, rounded as k_cgm_update_p does
template <class V2, typename R> struct PSource {
    const V2 *p, *r;
    R z, a;
    __device__ __forceinline__ V2 at(size_t i) const
    {
#pragma clang fp contract(off)
        const V2 pv = p[i], rv = r[i];
        return mk<V2>(fmadd(z, rv.x, a * pv.x), fmadd(z, rv.y, a * pv.y));
    }
};
template <bool AOS = false, class V2, typename R>
__device__ __forceinline__ void gather(const PSource<V2, R> &src, uint32_t n, uint32_t Vh, V2 v[3])
{
    static_assert(!AOS, "colour planes");
#pragma unroll
    for (int c = 0; c < 3; ++c)
        v[c] = src.at((size_t)c * Vh + n);
}

template <class A, class LK, int NR, int MU, int H, bool AOS = false, class Src>
__device__ __forceinline__ void hop_fwd(const A &a, const LK &lk, uint32_t s, const SiteCoord &sc,
                                        const Src *src, typename A::R acc[NR][6])
{
    using R = typename A::R;
    c2_t<R> U[9];
    lk.load(a.dst_parity, MU, s, U);
    const uint32_t n = nb_index<MU>(a.g, s, sc, H);
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        typename A::V2 v[3];
        gather<AOS>(src[j], n, a.g.Vh, v);
        umv_add(U, v, acc[j]);
    }
}

template <class A, class LK, int NR, int MU, int H, bool AOS = false, class Src>
__device__ __forceinline__ void hop_bwd(const A &a, const LK &lk, uint32_t s, const SiteCoord &sc,
                                        const Src *src, typename A::R acc[NR][6])
{
    using R = typename A::R;
    const uint32_t n = nb_index<MU>(a.g, s, sc, -H);
    c2_t<R> U[9];
    lk.load(1 - a.dst_parity, MU, n, U);
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        typename A::V2 v[3];
        gather<AOS>(src[j], n, a.g.Vh, v);
        udmv_sub(U, v, acc[j]);
    }
}

// Hop along x (MU 0) or y (MU 1) of a workgroup whose source rows are staged in LDS:
// st[j][c][k] holds colour c of right-hand side j at k = (y - y0 + 3) * Lx/2 + x/2 for the rows
// y0 - 3 .. y0 + NT / (Lx/2) + 2 of the workgroup's plane (yl = y - y0). Same arithmetic, in the
// same order, as hop_fwd / hop_bwd.
template <class A, class LK, int NR, int MU, int H, bool BWD, int KR>
__device__ __forceinline__ void hop_staged(const A &a, const LK &lk, uint32_t s, const SiteCoord &sc, int yl,
                                           const typename A::V2 (*st)[3][KR], typename A::R acc[NR][6])
{
    using R = typename A::R;
    constexpr int XH = kStageLxh;
    const int h = BWD ? -H : H;
    const int k = MU == 0 ? (yl + 3) * XH + (wrap_add(sc.c[0], h, a.g.L[0]) >> 1) : (yl + 3 + h) * XH + (sc.c[0] >> 1);
    c2_t<R> U[9];
    if (BWD)
        lk.load(1 - a.dst_parity, MU, nb_index<MU>(a.g, s, sc, h), U);
    else
        lk.load(a.dst_parity, MU, s, U);
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        typename A::V2 v[3];
#pragma unroll
        for (int c = 0; c < 3; ++c)
            v[c] = st[j][c][k];
        if (BWD)
            udmv_sub(U, v, acc[j]);
        else
            umv_add(U, v, acc[j]);
    }
}

// The staged kernel's 16 hops as one chain in which each hop's link words are requested before
// the previous hop's arithmetic (a one-hop prefetch; hop I: 0-3 x/y forward from LDS, 4-7 z/t
// forward from global memory, 8-11 and 12-15 the same backward; even I fat, odd I long links).
// A scheduling fence after each prefetch keeps the compiler from sinking it back. Measured at 32^4
// with FP32 links: 4 right-hand sides -2 %, 8 -8 %, 2 and 3 within 1 % (so used from 4 on, FP32
// links only: the FP64 link words would take 28-36 more registers).
template <int I> struct StagedHop {
    static constexpr int kMu = (I % 8) / 2;  // 0, 1 staged (x, y); 2, 3 global (z, t)
    static constexpr bool kBwd = I >= 8, kLong = (I % 2) == 1;
    static constexpr int kH = kLong ? 3 : 1;
};

template <class A, int I>
__device__ __forceinline__ auto staged_fetch(const A &a, uint32_t s, const SiteCoord &sc, uint32_t &n)
{
    using H = StagedHop<I>;
    n = nb_index<H::kMu>(a.g, s, sc, H::kBwd ? -H::kH : H::kH);
    const uint32_t ls = H::kBwd ? n : s;
    const int q = H::kBwd ? 1 - a.dst_parity : a.dst_parity;
    if constexpr (H::kLong)
        return a.lng.fetch(q, H::kMu, ls);
    else
        return a.fat.fetch(q, H::kMu, ls);
}

template <class A, int NR, int KR, int I, class RW>
__device__ __forceinline__ void staged_chain(const A &a, uint32_t s, const SiteCoord &sc, int yl,
                                             const typename A::V2 (*st)[3][KR], const typename A::V2 *const src[NR],
                                             typename A::R acc[NR][6], const RW &cur, uint32_t n)
{
    using H = StagedHop<I>;
    constexpr int XH = kStageLxh;
    typename A::V2 v[NR][3];
    if constexpr (H::kMu < 2) {
        const int h = H::kBwd ? -H::kH : H::kH;
        const int k = H::kMu == 0 ? (yl + 3) * XH + (wrap_add(sc.c[0], h, a.g.L[0]) >> 1)
                                  : (yl + 3 + h) * XH + (sc.c[0] >> 1);
#pragma unroll
        for (int j = 0; j < NR; ++j)
#pragma unroll
            for (int c = 0; c < 3; ++c)
                v[j][c] = st[j][c][k];
    } else {
#pragma unroll
        for (int j = 0; j < NR; ++j)
            gather(src[j], n, a.g.Vh, v[j]);
    }
    uint32_t n2 = 0;
    if constexpr (I < 15) {
        const auto nxt = staged_fetch<A, I + 1>(a, s, sc, n2);
        __builtin_amdgcn_sched_barrier(0);
        c2_t<typename A::R> U[9];
        if constexpr (H::kLong)
            a.lng.unpack(cur, U);
        else
            a.fat.unpack(cur, U);
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            if constexpr (H::kBwd)
                udmv_sub(U, v[j], acc[j]);
            else
                umv_add(U, v[j], acc[j]);
        }
        staged_chain<A, NR, KR, I + 1>(a, s, sc, yl, st, src, acc, nxt, n2);
    } else {
        c2_t<typename A::R> U[9];
        if constexpr (H::kLong)
            a.lng.unpack(cur, U);
        else
            a.fat.unpack(cur, U);
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            if constexpr (H::kBwd)
                udmv_sub(U, v[j], acc[j]);
            else
                umv_add(U, v[j], acc[j]);
        }
    }
}

// output store: streaming for the FP64 and FP32 link formats (measured 5% and 4%
// faster at 32^4), plain for the 16-bit one (3% slower with streaming stores). Also
// streaming where the next hopping term gathers the output (MdaggM's intermediate):
// plain stores there made the 32^4 solves 1-2% slower. The choice must stay
// compile-time: a run-time flag in this store made the FP64 term almost 2x slower.
template <class LF, class V2> __device__ __forceinline__ void put(V2 *p, V2 v)
{
    if constexpr (std::is_same<LF, LinkH>::value)
        *p = v;
    else
        st_nt(p, v);
}

// Entry of colour c of site s of a vector in colour planes or in the caller's host layout
template <bool AOS> __device__ __forceinline__ size_t entry_of(uint32_t Vh, uint32_t s, int c)
{
    return AOS ? (size_t)3 * s + c : (size_t)c * Vh + s;
}

// Epilogue of the hopping term: store D src (EPI_STORE), dst = sigma0 aux - D src with dst and aux
// in the caller's host layout (EPI_AXMY), or dst = sigma aux - D src with the per-workgroup partial
// sums of <aux, dst> (EPI_AXMY_DOT).
template <class LF, typename SR, int NR, int EPI, int NT, bool AOS = false, class A, typename R>
__device__ __forceinline__ void dslash_epilogue(const A &a, const R (&acc)[NR][6], c2_t<SR> *const (&dst)[NR],
                                                const c2_t<SR> *const (&aux)[NR], const int (&rr)[NR], int j0,
                                                int nact, uint32_t s, bool valid, double *lds)
{
    using V2 = c2_t<SR>;
    const uint32_t Vh = a.g.Vh;
    if constexpr (EPI == EPI_STORE) {
        if (valid) {
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                // padding slots repeat the last live right-hand side, so the
                // store is unconditional (same value to the same address)
                V2 o[3];
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    o[c] = mk<V2>((SR)acc[j][2 * c], (SR)acc[j][2 * c + 1]);
                if constexpr (AOS) {
                    st_site(dst[j] + (size_t)3 * s, o);
                } else {
#pragma unroll
                    for (int c = 0; c < 3; ++c)
                        put<LF>(&dst[j][(size_t)c * Vh + s], o[c]);
                }
            }
        }
    } else if constexpr (EPI == EPI_AXMY) {
        static_assert(NR == 1 && AOS, "the operator entry points' last term: one vector, host layout");
        if (valid) {
            V2 p[3], o[3];
            gather<true>(aux[0], s, Vh, p);
#pragma unroll
            for (int c = 0; c < 3; ++c)
                o[c] = mk<V2>((SR)((R)a.sigma0 * (R)p[c].x - acc[0][2 * c]),
                              (SR)((R)a.sigma0 * (R)p[c].y - acc[0][2 * c + 1]));
            st_site(dst[0] + (size_t)3 * s, o);
        }
    } else {
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            const bool live = j0 + j < nact;  // uniform over the block
            double d = 0.0;
            if (valid && live) {
                const double sg = a.sigma[rr[j]];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const V2 p = aux[j][(size_t)c * Vh + s];
                    const SR ox = (SR)((R)sg * (R)p.x - acc[j][2 * c]);
                    const SR oy = (SR)((R)sg * (R)p.y - acc[j][2 * c + 1]);
                    put<LF>(&dst[j][(size_t)c * Vh + s], mk<V2>(ox, oy));
                    d += (double)p.x * (double)ox + (double)p.y * (double)oy;
                }
            }
            const double tot = block_sum<NT>(d, lds);
            if (threadIdx.x == 0 && live)
                a.partial[(size_t)rr[j] * a.nblk + blockIdx.x] = tot;
            __syncthreads();
        }
    }
}

// Per right-hand-side base pointers of a workgroup's block of NR systems, resolved once (uniform
// over the block); padding slots beyond the nact live ones repeat the last live system
template <int NR, class A>
__device__ __forceinline__ void dslash_rhs(const A &a, int j0, int nact, int (&rr)[NR], typename A::V2 *(&dst)[NR],
                                           const typename A::V2 *(&src)[NR], const typename A::V2 *(&aux)[NR], bool with_aux)
{
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        const int jj = (j0 + j < nact) ? j0 + j : nact - 1;
        rr[j] = a.rlist ? a.rlist[jj] : jj;
        src[j] = a.src.p + a.src.base(rr[j]);
        dst[j] = a.dst.p + a.dst.base(rr[j]);
        aux[j] = with_aux ? a.aux.p + a.aux.base(rr[j]) : nullptr;
    }
}

template <class LF, class LL, typename SR, int NR, int EPI, int NT, int LAY = LAY_SOA>
__global__ void __launch_bounds__(NT) k_dslash(const DslashArgs<LF, LL, SR> a)
{
    using A = DslashArgs<LF, LL, SR>;
    using R = typename A::R;
    using V2 = c2_t<SR>;
    constexpr bool SA = (LAY & LAY_HOST_SRC) != 0, DA = (LAY & LAY_HOST_DST) != 0;
    __shared__ double lds[NT / kWave];
    if (a.run != nullptr && *a.run == 0)
        return;  // uniform over the grid
    const int nact = a.nact ? *a.nact : a.nrhs;
    const int j0 = blockIdx.y * NR;
    if (j0 >= nact)
        return;  // uniform over the block
    int rr[NR];
    const V2 *src[NR];
    V2 *dst[NR];
    const V2 *aux[NR];
    dslash_rhs<NR>(a, j0, nact, rr, dst, src, aux, EPI != EPI_STORE);
    bool valid;
    const uint32_t s = tile_site<NT>(a.g, blockIdx.x, gridDim.x, threadIdx.x, valid);
    R acc[NR][6];
#pragma unroll
    for (int j = 0; j < NR; ++j)
#pragma unroll
        for (int k = 0; k < 6; ++k)
            acc[j][k] = 0;
    if (valid) {
        const SiteCoord sc = site_coords(a.g, s, a.dst_parity);
        hop_fwd<A, LF, NR, 0, 1, SA>(a, a.fat, s, sc, src, acc);
        hop_fwd<A, LL, NR, 0, 3, SA>(a, a.lng, s, sc, src, acc);
        hop_fwd<A, LF, NR, 1, 1, SA>(a, a.fat, s, sc, src, acc);
        hop_fwd<A, LL, NR, 1, 3, SA>(a, a.lng, s, sc, src, acc);
        hop_fwd<A, LF, NR, 2, 1, SA>(a, a.fat, s, sc, src, acc);
        hop_fwd<A, LL, NR, 2, 3, SA>(a, a.lng, s, sc, src, acc);
        hop_fwd<A, LF, NR, 3, 1, SA>(a, a.fat, s, sc, src, acc);
        hop_fwd<A, LL, NR, 3, 3, SA>(a, a.lng, s, sc, src, acc);
        hop_bwd<A, LF, NR, 0, 1, SA>(a, a.fat, s, sc, src, acc);
        hop_bwd<A, LL, NR, 0, 3, SA>(a, a.lng, s, sc, src, acc);
        hop_bwd<A, LF, NR, 1, 1, SA>(a, a.fat, s, sc, src, acc);
        hop_bwd<A, LL, NR, 1, 3, SA>(a, a.lng, s, sc, src, acc);
        hop_bwd<A, LF, NR, 2, 1, SA>(a, a.fat, s, sc, src, acc);
        hop_bwd<A, LL, NR, 2, 3, SA>(a, a.lng, s, sc, src, acc);
        hop_bwd<A, LF, NR, 3, 1, SA>(a, a.fat, s, sc, src, acc);
        hop_bwd<A, LL, NR, 3, 3, SA>(a, a.lng, s, sc, src, acc);
    }
    dslash_epilogue<LF, SR, NR, EPI, NT, DA>(a, acc, dst, aux, rr, j0, nact, s, valid, lds);
}

// ---- split hopping term: S waves per 64 sites, each with 16 / S of the 16 hops
//
// With one thread per site a small lattice leaves most of the chip idle (8^4 has 2048 sites of one
// parity: 32 waves on 1024 SIMDs) and each wave walks a serial chain of 16 link and neighbour
// loads, so the time is latency. Here the S waves of a workgroup take the hops of the same 64
// sites, keep the links' coalesced loads (lane = site) and add their partial results through LDS,
// in wave order: S times the waves in flight and 1/S of the chain. Consecutive threads then own
// consecutive entries of the destination's layout, so the host layout is written coalesced.
// Measured per FP64 term (LinkD, LinkD14, one right-hand side), one thread per site in workgroups
// of 256 -> S = 8: 8^4 8.9 -> 4.5 us, 12^4 16.5 -> 6.8, 16^4 18.9 -> 12.4, 22x18x15x13
// 20.6 -> 17.1; at 16^3x32 and above, where the one-thread form fills the chip, up to 10 % slower
// (32^4 176 -> 195). S = 4 and 16 are up to 10 % slower than 8 at 8^4 to 16^4.

// Hops of one wave: hop I = 4 mu + 2 (backward) + (3 hops)
template <class A, class LF, class LL, int NR, bool SA, int I, class Src>
__device__ __forceinline__ void split_hop(const A &a, uint32_t s, const SiteCoord &sc, const Src *src,
                                          typename A::R acc[NR][6])
{
    constexpr int MU = I / 4;
    if constexpr ((I & 3) == 0)
        hop_fwd<A, LF, NR, MU, 1, SA>(a, a.fat, s, sc, src, acc);
    else if constexpr ((I & 3) == 1)
        hop_fwd<A, LL, NR, MU, 3, SA>(a, a.lng, s, sc, src, acc);
    else if constexpr ((I & 3) == 2)
        hop_bwd<A, LF, NR, MU, 1, SA>(a, a.fat, s, sc, src, acc);
    else
        hop_bwd<A, LL, NR, MU, 3, SA>(a, a.lng, s, sc, src, acc);
}

template <class A, class LF, class LL, int NR, bool SA, int I, int N, class Src>
__device__ __forceinline__ void split_hops(const A &a, uint32_t s, const SiteCoord &sc, const Src *src,
                                           typename A::R acc[NR][6])
{
    split_hop<A, LF, LL, NR, SA, I>(a, s, sc, src, acc);
    if constexpr (N > 1)
        split_hops<A, LF, LL, NR, SA, I + 1, N - 1>(a, s, sc, src, acc);
}

// Each wave branches on its index, a value uniform over the wave, to code of its own. The network's
// layers in that form were compiled wrongly (dir_neighbours in kq_ptnet.hip): the 64 weights that
// each path takes from the kernel's arguments filled the scalar registers, and a path was left with
// another one's. What a path here has in scalar registers of its own are link strides. None of these
// kernels may spill a scalar register (tests/test_kernel_resources.py); in the listing of each, walked
// for every wave index, no register is read and no address formed before it is written; and since no
// branch between the waves depends on data, the tests, which run every instantiation against
// the oracle, run all of its paths.
template <class A, class LF, class LL, int NR, bool SA, int S, int W, class Src>
__device__ __forceinline__ void split_wave(int w, const A &a, uint32_t s, const SiteCoord &sc, const Src *src,
                                           typename A::R acc[NR][6])
{
    if (w == W)
        split_hops<A, LF, LL, NR, SA, W * (16 / S), 16 / S>(a, s, sc, src, acc);
    else if constexpr (W + 1 < S)
        split_wave<A, LF, LL, NR, SA, S, W + 1>(w, a, s, sc, src, acc);
}

template <class LF, class LL, typename SR, int NR, int EPI, int S, int LAY = LAY_SOA>
__global__ void __launch_bounds__(64 * S) k_dslash_split(const DslashArgs<LF, LL, SR> a)
{
    using A = DslashArgs<LF, LL, SR>;
    using R = typename A::R;
    using V2 = c2_t<SR>;
    constexpr bool SA = (LAY & LAY_HOST_SRC) != 0, DA = (LAY & LAY_HOST_DST) != 0;
    constexpr int NT = 64 * S;
    // results of half the waves: the other half adds its own to them, so that the workgroup's LDS is
    // half of one slot per wave (blocks of 8 FP32 right-hand sides: 24.6 instead of 49 KB, 4
    // instead of 3 workgroups per CU; LinkF + LinkF12 16^3x32 35.6 -> 30.3 us, 32^4 213 -> 203)
    constexpr int H = S / 2, DOTS = EPI == EPI_AXMY_DOT ? NR : 1;
    __shared__ R red[H][NR][6][64];
    __shared__ uint32_t site[64];
    __shared__ double lds[S][DOTS];
    if (a.run != nullptr && *a.run == 0)
        return;  // uniform over the grid
    const int nact = a.nact ? *a.nact : a.nrhs;
    const int j0 = blockIdx.y * NR;
    if (j0 >= nact)
        return;  // uniform over the block
    int rr[NR];
    const V2 *src[NR];
    V2 *dst[NR];
    const V2 *aux[NR];
    dslash_rhs<NR>(a, j0, nact, rr, dst, src, aux, EPI != EPI_STORE);
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t Vh = a.g.Vh;
    bool valid;
    const uint32_t s = tile_site<64>(a.g, blockIdx.x, gridDim.x, lane, valid);
    R acc[NR][6];
#pragma unroll
    for (int j = 0; j < NR; ++j)
#pragma unroll
        for (int k = 0; k < 6; ++k)
            acc[j][k] = 0;
    if (valid) {
        const SiteCoord sc = site_coords(a.g, s, a.dst_parity);
        split_wave<A, LF, LL, NR, SA, S, 0>(w, a, s, sc, src, acc);
    }
    if (w == 0)
        site[lane] = valid ? s : 0xffffffffu;
    if (w >= H) {
#pragma unroll
        for (int j = 0; j < NR; ++j)
#pragma unroll
            for (int k = 0; k < 6; ++k)
                red[w - H][j][k][lane] = acc[j][k];
    }
    __syncthreads();
    if (w < H) {
#pragma unroll
        for (int j = 0; j < NR; ++j)
#pragma unroll
            for (int k = 0; k < 6; ++k)
                red[w][j][k][lane] += acc[j][k];
    }
    __syncthreads();
    if constexpr (NR == 8 && EPI == EPI_AXMY_DOT) {
        // The epilogue's pointers are resolved again: kept across the waves' hops, 24 of them spilled
        // scalar registers there (split_wave). The empty asm makes the block's index unknown to the
        // compiler, which would keep the first ones otherwise.
        uint32_t y = blockIdx.y;
        asm("" : "+s"(y));
        dslash_rhs<NR>(a, (int)y * NR, nact, rr, dst, src, aux, true);
    }
    // 192 complex results per right-hand side, summed over the slots in their order; consecutive
    // threads take consecutive entries of the destination's layout
    double d[DOTS];
#pragma unroll
    for (int j = 0; j < DOTS; ++j)
        d[j] = 0.0;
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        if (j0 + j >= nact)
            continue;  // uniform over the block
        for (int e = threadIdx.x; e < 192; e += NT) {
            const int l = DA ? e / 3 : (e & 63), c = DA ? e - 3 * l : e >> 6;
            const uint32_t sl = site[l];
            if (sl == 0xffffffffu)
                continue;
            R x = red[0][j][2 * c][l], y = red[0][j][2 * c + 1][l];
#pragma unroll
            for (int k = 1; k < H; ++k) {
                x += red[k][j][2 * c][l];
                y += red[k][j][2 * c + 1][l];
            }
            const size_t o = entry_of<DA>(Vh, sl, c);
            V2 v = mk<V2>((SR)x, (SR)y);
            if constexpr (EPI != EPI_STORE) {
                const R sg = (R)(EPI == EPI_AXMY ? a.sigma0 : a.sigma[rr[j]]);
                const V2 p = DA ? ld_u(&aux[j][o]) : aux[j][o];
                v = mk<V2>((SR)(sg * (R)p.x - x), (SR)(sg * (R)p.y - y));
                if constexpr (EPI == EPI_AXMY_DOT)
                    d[j] += (double)p.x * (double)v.x + (double)p.y * (double)v.y;
            }
            if constexpr (DA)
                st_u(&dst[j][o], v);
            else
                put<LF>(&dst[j][o], v);
        }
    }
    if constexpr (EPI == EPI_AXMY_DOT) {
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            const double v = wave_sum(d[j]);
            if (lane == 0)
                lds[w][j] = v;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NR; ++j)
            if (threadIdx.x == j && j0 + j < nact) {
                double tot = 0.0;
#pragma unroll
                for (int k = 0; k < S; ++k)
                    tot += lds[k][j];
                a.partial[(size_t)rr[j] * a.nblk + blockIdx.x] = tot;
            }
    }
}

// The split hopping term of one system, deferred or down to one shift, with the previous iteration's
// direction update on the way: src is p before the update, every gather forms z r + a p, and the
// workgroup stores the updated direction of its own 64 entries in pnew (two buffers take turns: other
// workgroups still gather the old one) and, if the system is not deferred, their solution. An iteration
// then has 3 kernels instead of 4, which is what a small lattice's time consists of; the gathers
// double, from L2. The last workgroup finishes the previous iteration's scalars instead, and every
// workgroup adds the npart partials of |r|^2 wave by wave in the same order.
// Per launch (LinkD, LinkD14, 8^4) 6.4 us against 5.1 for the plain term and 3.7 for the update; at
// 16^4 in FP32 10.9 against 8.8 and 4.2. Bound by its chain of loads and by the launch itself.
template <class LF, class LL, typename SR>
__global__ void __launch_bounds__(512)
k_dslash_split_p(const DslashArgs<LF, LL, SR> a, CgmState<SR> *st, const c2_t<SR> *r, Vec<SR> pnew, Vec<SR> x,
                 const double *part, uint32_t npart, double *shist)
{
    using A = DslashArgs<LF, LL, SR>;
    using V2 = c2_t<SR>;
    constexpr int S = 8, H = S / 2, NT = 64 * S;
    __shared__ SR red[H][1][6][64];
    __shared__ uint32_t site[64];
    if (st->run == 0)
        return;  // uniform over the grid: no workgroup of this kernel writes it
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double l2 = 0.0;
    for (uint32_t i = lane; i < npart; i += 64)
        l2 += part[i];
    l2 = wave_sum(l2);
    if (blockIdx.x == a.nblk) {
        cgm_finish_iteration(*st, l2, shist);
        return;
    }
    const PSource<V2, SR> src{a.src.p + a.src.base(0), r, st->Z[0], (SR)l2 / st->rr_prev};
    bool valid;
    const uint32_t s = tile_site<64>(a.g, blockIdx.x, a.nblk, lane, valid);
    SR acc[1][6];
#pragma unroll
    for (int k = 0; k < 6; ++k)
        acc[0][k] = 0;
    if (valid) {
        const SiteCoord sc = site_coords(a.g, s, a.dst_parity);
        split_wave<A, LF, LL, 1, false, S, 0>(w, a, s, sc, &src, acc);
    }
    if (w == 0)
        site[lane] = valid ? s : 0xffffffffu;
    if (w >= H) {
#pragma unroll
        for (int k = 0; k < 6; ++k)
            red[w - H][0][k][lane] = acc[0][k];
    }
    __syncthreads();
    if (w < H) {
#pragma unroll
        for (int k = 0; k < 6; ++k)
            red[w][0][k][lane] += acc[0][k];
    }
    __syncthreads();
    const int e = threadIdx.x - (NT - 192);  // the last three waves store one colour each
    if (e < 0)
        return;
    const int l = e & 63, c = e >> 6;
    const uint32_t sl = site[l];
    if (sl == 0xffffffffu)
        return;
    SR re = red[0][0][2 * c][l], im = red[0][0][2 * c + 1][l];
#pragma unroll
    for (int k = 1; k < H; ++k) {
        re += red[k][0][2 * c][l];
        im += red[k][0][2 * c + 1][l];
    }
    const size_t o = (size_t)c * a.g.Vh + sl;
    put<LF>(&a.dst.p[a.dst.base(0) + o], mk<V2>(re, im));
    pnew.p[pnew.base(0) + o] = src.at(o);
    if (st->dslot < 0) {
        const SR b = st->B[0];
        const V2 po = src.p[o];
        V2 *xo = x.p + x.base(0) + o, xv = *xo;
        xv.x = fmadd(-b, po.x, xv.x);
        xv.y = fmadd(-b, po.y, xv.y);
        *xo = xv;
    }
}

template <class LF, class LL, typename SR>
void launch_dslash_p(DslashArgs<LF, LL, SR> a, CgmState<SR> *st, const c2_t<SR> *r, Vec<SR> pnew, Vec<SR> x,
                     const double *part, uint32_t npart, double *shist, hipStream_t stream)
{
    if (a.nrhs != 1 || dslash_split_waves(std::is_same<SR, double>::value, a.g, 1, 1) != 8)
        throw std::logic_error("dslash: the direction update needs one system and the split term of 8 waves");
    a.nblk = dslash_grid(a.g.Vh, 64);
    hipLaunchKernelGGL((k_dslash_split_p<LF, LL, SR>), dim3(a.nblk + 1), dim3(512), 0, stream, a, st, r, pnew, x,
                       part, npart, shist);
    KQ_HIP_CHECK(hipGetLastError());
}

// The batched hopping term with the x and y neighbours read from LDS: the workgroup (256 sites,
// whole x-rows of one (x, y) plane, stage_rows()) first copies its rows and their +-3
// y-neighbour rows of every source into LDS; the z and t neighbours come from global memory.
// Used for NR >= 2, where every staged row serves several right-hand sides' gathers: measured at
// 32^4 with FP32 links, 4 right-hand sides 130 -> 116 us, 2 and 8 about 4 % faster (1 would be
// a little slower). Results are bitwise those of k_dslash.
template <class LF, class LL, typename SR, int NR, int EPI>
__global__ void __launch_bounds__(256) k_dslash_staged(const DslashArgs<LF, LL, SR> a)
{
    using A = DslashArgs<LF, LL, SR>;
    using R = typename A::R;
    using V2 = c2_t<SR>;
    constexpr int NT = 256, XH = kStageLxh, KR = NT + 6 * XH;
    __shared__ __align__(16) V2 st[NR][3][KR];
    __shared__ double lds[NT / kWave];
    if (a.run != nullptr && *a.run == 0)
        return;  // uniform over the grid
    const int nact = a.nact ? *a.nact : a.nrhs;
    const int j0 = blockIdx.y * NR;
    if (j0 >= nact)
        return;  // uniform over the block
    int rr[NR];
    const V2 *src[NR];
    V2 *dst[NR];
    const V2 *aux[NR];
    dslash_rhs<NR>(a, j0, nact, rr, dst, src, aux, EPI == EPI_AXMY_DOT);
    const uint32_t Vh = a.g.Vh;
    // true for every thread where this kernel is launched (tile order); the hops and the epilogue
    // stay under it as in k_dslash: with the hops outside, the compiler moved them into the
    // epilogue's branches and used twice the registers, with spills
    bool valid;
    const uint32_t s = tile_site<NT>(a.g, blockIdx.x, gridDim.x, threadIdx.x, valid);
    const SiteCoord sc = site_coords(a.g, s, a.dst_parity);
    const int yl = (int)threadIdx.x / XH;
    const int y0 = sc.c[1] - yl;  // uniform over the workgroup
    const uint32_t pbase = s - threadIdx.x - (uint32_t)(XH * y0);
    const int L1 = a.g.L[1];
    // rows are XH entries of one colour plane, so two FP32 entries (16 bytes) load together when
    // every source is 16-byte aligned (Vh even: so are its colour planes and rows)
    bool wide = sizeof(V2) == 8 && (Vh % 2u) == 0;
#pragma unroll
    for (int j = 0; j < NR; ++j)
        wide = wide && ((reinterpret_cast<uintptr_t>(src[j]) & 15u) == 0);
    if (wide) {
        constexpr int KH = KR / 2;
        for (int e = threadIdx.x; e < NR * 3 * KH; e += NT) {
            const int jc = e / KH, kk = 2 * (e - jc * KH), j = jc / 3, c = jc - 3 * j;
            const int row = kk / XH, xh = kk - row * XH;
            int ys = y0 - 3 + row;
            ys = ys < 0 ? ys + L1 : (ys >= L1 ? ys - L1 : ys);
            const uint32_t n = pbase + (uint32_t)(XH * ys + xh);
            *reinterpret_cast<kq_v4f *>(&st[j][c][kk]) =
                *reinterpret_cast<const kq_v4f *>(a.src.p + a.src.base(rr[j]) + (size_t)c * Vh + n);
        }
    } else {
        for (int e = threadIdx.x; e < NR * 3 * KR; e += NT) {
            const int jc = e / KR, kk = e - jc * KR, j = jc / 3, c = jc - 3 * j;
            const int row = kk / XH, xh = kk - row * XH;
            int ys = y0 - 3 + row;
            ys = ys < 0 ? ys + L1 : (ys >= L1 ? ys - L1 : ys);
            const uint32_t n = pbase + (uint32_t)(XH * ys + xh);
            st[j][c][kk] = a.src.p[a.src.base(rr[j]) + (size_t)c * Vh + n];
        }
    }
    __syncthreads();
    R acc[NR][6];
#pragma unroll
    for (int j = 0; j < NR; ++j)
#pragma unroll
        for (int k = 0; k < 6; ++k)
            acc[j][k] = 0;
    if (valid) {
        if constexpr (NR >= 4 && std::is_same<R, float>::value) {
            uint32_t n0;
            const auto r0 = staged_fetch<A, 0>(a, s, sc, n0);
            staged_chain<A, NR, KR, 0>(a, s, sc, yl, st, src, acc, r0, n0);
        } else {
            hop_staged<A, LF, NR, 0, 1, false, KR>(a, a.fat, s, sc, yl, st, acc);
            hop_staged<A, LL, NR, 0, 3, false, KR>(a, a.lng, s, sc, yl, st, acc);
            hop_staged<A, LF, NR, 1, 1, false, KR>(a, a.fat, s, sc, yl, st, acc);
            hop_staged<A, LL, NR, 1, 3, false, KR>(a, a.lng, s, sc, yl, st, acc);
            hop_fwd<A, LF, NR, 2, 1>(a, a.fat, s, sc, src, acc);
            hop_fwd<A, LL, NR, 2, 3>(a, a.lng, s, sc, src, acc);
            hop_fwd<A, LF, NR, 3, 1>(a, a.fat, s, sc, src, acc);
            hop_fwd<A, LL, NR, 3, 3>(a, a.lng, s, sc, src, acc);
            hop_staged<A, LF, NR, 0, 1, true, KR>(a, a.fat, s, sc, yl, st, acc);
            hop_staged<A, LL, NR, 0, 3, true, KR>(a, a.lng, s, sc, yl, st, acc);
            hop_staged<A, LF, NR, 1, 1, true, KR>(a, a.fat, s, sc, yl, st, acc);
            hop_staged<A, LL, NR, 1, 3, true, KR>(a, a.lng, s, sc, yl, st, acc);
            hop_bwd<A, LF, NR, 2, 1>(a, a.fat, s, sc, src, acc);
            hop_bwd<A, LL, NR, 2, 3>(a, a.lng, s, sc, src, acc);
            hop_bwd<A, LF, NR, 3, 1>(a, a.fat, s, sc, src, acc);
            hop_bwd<A, LL, NR, 3, 3>(a, a.lng, s, sc, src, acc);
        }
    }
    dslash_epilogue<LF, SR, NR, EPI, NT>(a, acc, dst, aux, rr, j0, nact, s, valid, lds);
}

// LDS of a workgroup the device allows
static int lds_block_bytes()
{
    static const int lds_block = [] {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v <= 0)
            v = 65536;
        return v;
    }();
    return lds_block;
}

// dynamic LDS bytes that let at most `cap` waves per SIMD (4 SIMDs per CU) be resident
static size_t cap_lds_bytes(int cap, int nt)
{
    if (cap <= 0)
        return 0;
    static const int lds_cu = [] {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) != hipSuccess || v <= 0)
            v = 65536;
        return v;
    }();
    const int lds_block = lds_block_bytes();
    const int blocks = std::max(1, cap * 4 / std::max(1, nt / kWave));
    // a little under lds_cu / blocks, so that `blocks` fit and blocks + 1 do not
    const int bytes = lds_cu / blocks - 256;
    return (size_t)std::max(0, std::min(bytes, lds_block - 256));
}

template <class LF, class LL, typename SR, int NR, int EPI>
static void launch_nt(const DslashArgs<LF, LL, SR> &a, int kernel, int nt, int cap, hipStream_t st)
{
    const int nact_max = a.nrhs;
    const dim3 grid(a.nblk, (nact_max + NR - 1) / NR);
    const size_t lds = cap_lds_bytes(cap, nt);
    if constexpr (NR >= 2) {
        // staged rows (static LDS of the kernel): NR * 3 colour entries for each of the
        // nt + 6 Lx/2 sites of the workgroup's rows and their +-3 y-neighbour rows; an occupancy
        // cap adds dynamic LDS only beyond that
        const size_t sb = (size_t)NR * 3 * (256 + 6 * kStageLxh) * sizeof(c2_t<SR>);
        if (kernel == kHopStaged && sb + 1024 <= (size_t)lds_block_bytes()) {
            hipLaunchKernelGGL((k_dslash_staged<LF, LL, SR, NR, EPI>), grid, dim3(256), lds > sb ? lds - sb : 0,
                               st, a);
            KQ_HIP_CHECK(hipGetLastError());
            return;
        }
    }
    switch (nt) {
    case 64:
        hipLaunchKernelGGL((k_dslash<LF, LL, SR, NR, EPI, 64>), grid, dim3(64), lds, st, a);
        break;
    case 128:
        hipLaunchKernelGGL((k_dslash<LF, LL, SR, NR, EPI, 128>), grid, dim3(128), lds, st, a);
        break;
    default:
        hipLaunchKernelGGL((k_dslash<LF, LL, SR, NR, EPI, 256>), grid, dim3(256), lds, st, a);
        break;
    }
    KQ_HIP_CHECK(hipGetLastError());
}

template <class LF, class LL, typename SR, int NR, int S>
static void launch_split(const DslashArgs<LF, LL, SR> &a, int epi, hipStream_t st)
{
    const dim3 grid(a.nblk, (a.nrhs + NR - 1) / NR), blk(64 * S);
    if (epi == EPI_STORE)
        hipLaunchKernelGGL((k_dslash_split<LF, LL, SR, NR, EPI_STORE, S>), grid, blk, 0, st, a);
    else
        hipLaunchKernelGGL((k_dslash_split<LF, LL, SR, NR, EPI_AXMY_DOT, S>), grid, blk, 0, st, a);
    KQ_HIP_CHECK(hipGetLastError());
}

template <class LF, class LL, typename SR, int NR>
static uint32_t launch_epi(DslashArgs<LF, LL, SR> a, int epi, int nt, int cap, hipStream_t st)
{
    constexpr bool kDouble = std::is_same<SR, double>::value;
    constexpr bool kSmallLong = LL::kBytes < 40;
    const int kernel = hop_kernel(kDouble, kSmallLong, a.g, a.nrhs, NR, nt);
    if (kernel > kHopStaged)
        a.nblk = dslash_grid(a.g.Vh, 64);
    if constexpr (!kDouble || NR <= 2) {
        constexpr int S = NR <= 2 ? 8 : 4;
        if (kernel == S) {
            launch_split<LF, LL, SR, NR, S>(a, epi, st);
            return a.nblk;
        }
    }
    if constexpr (NR == 8 && kSmallLong) {
        if (kernel == 2) {
            launch_split<LF, LL, SR, NR, 2>(a, epi, st);
            return a.nblk;
        }
    }
    a.nblk = dslash_grid(a.g.Vh, nt);
    if (epi == EPI_STORE)
        launch_nt<LF, LL, SR, NR, EPI_STORE>(a, kernel, nt, cap, st);
    else
        launch_nt<LF, LL, SR, NR, EPI_AXMY_DOT>(a, kernel, nt, cap, st);
    return a.nblk;
}

// Hopping term on the caller's host layout (kq_dslash.h)
template <class LF, class LL, typename SR, int NR, int S>
static void launch_host_split(DslashArgs<LF, LL, SR> a, int lay, int epi, hipStream_t st)
{
    a.nblk = dslash_grid(a.g.Vh, 64);
    const dim3 grid(a.nblk, (a.nrhs + NR - 1) / NR), blk(64 * S);
    if (lay == LAY_HOST && epi == EPI_STORE)
        hipLaunchKernelGGL((k_dslash_split<LF, LL, SR, NR, EPI_STORE, S, LAY_HOST>), grid, blk, 0, st, a);
    else if constexpr (NR == 1) {
        if (lay == LAY_HOST_SRC && epi == EPI_STORE)
            hipLaunchKernelGGL((k_dslash_split<LF, LL, SR, 1, EPI_STORE, S, LAY_HOST_SRC>), grid, blk, 0, st, a);
        else if (lay == LAY_HOST_DST && epi == EPI_AXMY)
            hipLaunchKernelGGL((k_dslash_split<LF, LL, SR, 1, EPI_AXMY, S, LAY_HOST_DST>), grid, blk, 0, st, a);
        else
            throw std::logic_error("dslash: unsupported layout");
    } else
        throw std::logic_error("dslash: unsupported layout");
    KQ_HIP_CHECK(hipGetLastError());
}

template <class LF, class LL, typename SR, int NT>
static void launch_host_nt(DslashArgs<LF, LL, SR> a, int lay, int epi, hipStream_t st)
{
    a.nblk = dslash_grid(a.g.Vh, NT);
    if (lay == LAY_HOST_SRC && epi == EPI_STORE)
        hipLaunchKernelGGL((k_dslash<LF, LL, SR, 1, EPI_STORE, NT, LAY_HOST_SRC>), dim3(a.nblk), dim3(NT), 0, st, a);
    else if (lay == LAY_HOST_DST && epi == EPI_AXMY)
        hipLaunchKernelGGL((k_dslash<LF, LL, SR, 1, EPI_AXMY, NT, LAY_HOST_DST>), dim3(a.nblk), dim3(NT), 0, st, a);
    else
        throw std::logic_error("dslash: unsupported layout");
    KQ_HIP_CHECK(hipGetLastError());
}

// Source in colour planes, destination in the host layout, one thread per site and block of NR vectors
template <class LF, class LL, typename SR, int NR>
static void launch_host_block(DslashArgs<LF, LL, SR> a, hipStream_t st)
{
    a.nblk = dslash_grid(a.g.Vh, 256);
    hipLaunchKernelGGL((k_dslash<LF, LL, SR, NR, EPI_STORE, 256, LAY_HOST_DST>), dim3(a.nblk, (a.nrhs + NR - 1) / NR),
                       dim3(256), 0, st, a);
    KQ_HIP_CHECK(hipGetLastError());
}

template <class LF, class LL, typename SR>
void launch_dslash_host(const DslashArgs<LF, LL, SR> &a, int lay, int epi, int nr, hipStream_t st)
{
    constexpr bool kDouble = std::is_same<SR, double>::value;
    if (a.g.Vh == 0 || a.nrhs <= 0)
        return;
    if (lay == LAY_HOST) {
        // Source and destination in the host layout: the split form at every size. Its epilogue
        // writes the 48- or 24-byte sites coalesced, where one thread per site writes them in
        // strides. Per launch, one thread per site -> split: FP64, one right-hand side, 24^4
        // 67.6 -> 65 us, 32^4 206 -> 196, 48^4 1087 -> 1015; FP32, 8 right-hand sides in blocks of
        // 4, 24^4 110 -> 82, 48^4 1597 -> 1382; in one block of 8 (S = 4), 24^4 90 -> 63. FP64
        // blocks above 2 spill, so larger ones run as blocks of 2 (or not here: host_planes_block).
        if constexpr (kDouble) {
            if (nr >= 2)
                launch_host_split<LF, LL, SR, 2, 8>(a, lay, epi, st);
            else
                launch_host_split<LF, LL, SR, 1, 8>(a, lay, epi, st);
        } else {
            // Blocks of 4 of more than 4 vectors would read the links twice: above 16384 sites they run
            // as blocks of 8 (calls with 8 vectors in blocks of 4 -> 8, LinkF + LinkF12: 16^4
            // 29.1 -> 26.3 us, 16^3x32 45.5 -> 42.7, 24^4 92.6 -> 76.1, 32^4 259 -> 198, 48^4
            // 1364 -> 981; with 5 vectors 27.4 -> 25.6 to 1238 -> 853; LinkF12C likewise; but 12^4
            // 20.7 -> 21.8, 8^4 16.8 -> 19.5)
            if (nr == 4 && a.nrhs > 4 && a.g.Vh > 16384u)
                nr = 8;
            switch (nr) {
            case 1:
                launch_host_split<LF, LL, SR, 1, 8>(a, lay, epi, st);
                break;
            case 2:
                launch_host_split<LF, LL, SR, 2, 8>(a, lay, epi, st);
                break;
            case 3:
                launch_host_split<LF, LL, SR, 3, 8>(a, lay, epi, st);
                break;
            case 4:
                launch_host_split<LF, LL, SR, 4, 8>(a, lay, epi, st);
                break;
            case 8:
                launch_host_split<LF, LL, SR, 8, 4>(a, lay, epi, st);
                break;
            default:
                throw std::runtime_error("dslash: unsupported RHS blocking " + std::to_string(nr));
            }
        }
        return;
    }
    if constexpr (kDouble) {
        if (lay == LAY_HOST_DST && epi == EPI_STORE) {
            if (nr == 3)
                launch_host_block<LF, LL, SR, 3>(a, st);
            else if (nr == 4)
                launch_host_block<LF, LL, SR, 4>(a, st);
            else
                launch_host_block<LF, LL, SR, 8>(a, st);
            return;
        }
    }
    // One side in the host layout (A = sigma - D D, one right-hand side): split up to the size at
    // which one thread per site fills the chip, measured per term, one thread -> split: FP64
    // 22x18x15x13 18.6 -> 16.9 us, 20^4 39.4 -> 31.7 (but 29.4 in workgroups of 64), 24^4
    // 61.4 -> 63.6, 32^4 182 -> 196; FP32 16^3x32 14.2 -> 12.2, 20^4 18.9 -> 15.7, 24^4
    // 29.4 -> 30.2. Workgroups of 64 below 200 000 sites, where a grid of 256-thread ones ends in
    // a partly filled round (24^4 64.4 -> 61.4 us; equal at 32^3x16).
    if (a.g.Vh <= (kDouble ? 49152u : 98304u))
        launch_host_split<LF, LL, SR, 1, 8>(a, lay, epi, st);
    else if (a.g.Vh < 200000u)
        launch_host_nt<LF, LL, SR, 64>(a, lay, epi, st);
    else
        launch_host_nt<LF, LL, SR, 256>(a, lay, epi, st);
}

template <class LF, class LL, typename SR>
uint32_t launch_dslash(DslashArgs<LF, LL, SR> a, int epi, int nr, int nt, hipStream_t st, int cap)
{
    if (a.g.Vh == 0 || a.nrhs <= 0)
        return 0;
    check_blocking(nr, nt);
    switch (nr) {
    case 1:
        return launch_epi<LF, LL, SR, 1>(a, epi, nt, cap, st);
    case 2:
        return launch_epi<LF, LL, SR, 2>(a, epi, nt, cap, st);
    case 3:
        return launch_epi<LF, LL, SR, 3>(a, epi, nt, cap, st);
    case 4:
        return launch_epi<LF, LL, SR, 4>(a, epi, nt, cap, st);
    default:
        return launch_epi<LF, LL, SR, 8>(a, epi, nt, cap, st);
    }
}

}  // namespace kq
