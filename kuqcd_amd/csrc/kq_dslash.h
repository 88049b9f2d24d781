// Host-side interface of the HISQ even-odd hopping-term kernels.
#pragma once

#include "kq_fields.h"

namespace kq {

enum DslashEpilogue {
    EPI_STORE = 0,     // dst = D src
    EPI_AXMY_DOT = 1,  // dst = sigma[r] * aux - D src ; partial[r][blk] = Re<aux, dst>
    EPI_AXMY = 2,      // dst = sigma0 * aux - D src (operator entry points)
};

// Layout of a hopping term's vectors: the library's colour planes, or the caller's host layout
// (v[3 s + c]) for the source (bit 0) or for the destination and aux (bit 1)
enum DslashLayout { LAY_SOA = 0, LAY_HOST_SRC = 1, LAY_HOST_DST = 2, LAY_HOST = 3 };

template <class LF, class LL, typename SR> struct DslashArgs {
    using R = typename LF::R;
    using V2 = c2_t<SR>;
    Geom g;
    int dst_parity;
    LF fat;
    LL lng;
    Vec<SR> src, dst, aux;
    const double *sigma;  // per right-hand side (EPI_AXMY_DOT)
    double sigma0;        // for every right-hand side (EPI_AXMY)
    double *partial;      // [nrhs_total][nblk] (EPI_AXMY_DOT)
    const int *run;       // device flag; kernel does nothing when *run == 0 (may be null)
    const int *rlist;     // compact list of active right-hand sides (may be null = identity)
    const int *nact;      // number of entries of rlist in use (may be null = nrhs)
    int nrhs;             // right-hand sides addressed by this launch
    uint32_t nblk;        // grid.x, the partial-sum stride
};

// block sizes launch_dslash accepts: 64, 128 and 256 threads
constexpr int kMinDslashNT = 64;
// Most sites of one parity (times the blocks of vectors) for which the split hopping term is the rule
// (dslash_split_waves), in FP64 and FP32
constexpr uint32_t kSplitSites64 = 49152, kSplitSites32 = 98304;
// Block size of the hopping terms whose partial sums feed the reference method, the plain
// FP64 solve and the FP64 verification. One partial per workgroup, added in a fixed order,
// makes a reduction deterministic for a given block size; fixing the block size by the lattice
// (instead of taking the autotuner's timing-dependent pick) makes these results bitwise
// reproducible from one process to the next. Below 200 000 sites a grid of 256-thread workgroups
// ends in a partly filled round (FP64 term at 20^4: 313 workgroups on 256 CUs, 37 us against 29 in
// workgroups of 64; 24^4 62 against 59.5); above, 256 is 1-3 % faster (32^4 176 against 181 us).
inline int repro_nt(uint32_t Vh) { return Vh < 200000u ? 64 : 256; }

// Blockings and block sizes that exist; others are refused on every lattice, also where the kernel
// that runs has a block size of its own
inline void check_blocking(int nr, int nt)
{
    if (nr != 1 && nr != 2 && nr != 3 && nr != 4 && nr != 8)
        throw std::runtime_error("dslash: unsupported RHS blocking " + std::to_string(nr));
    if (nt != 64 && nt != 128 && nt != 256)
        throw std::runtime_error("dslash: unsupported block size " + std::to_string(nt));
}

// Launch D over all sites of parity dst_parity for every right-hand side.
// nr = right-hand sides handled per thread (1, 2, 3, 4 or 8), nt = threads per block,
// cap = at most this many wavefronts per SIMD (0: as many as the registers allow). The
// cap is imposed with unused dynamic LDS; fewer resident waves keep the gathered
// neighbour vectors of the batched terms in L2 (measured up to 19 % faster at 32^4). Where the
// split or the LDS-staged kernel runs, nt (and for the split one cap) has no effect.
// Returns the number of workgroups over the sites: the stride of the partial sums per right-hand
// side, at most dslash_nblk(Vh, kMinDslashNT).
template <class LF, class LL, typename SR>
uint32_t launch_dslash(DslashArgs<LF, LL, SR> a, int epi, int nr, int nt, hipStream_t st, int cap = 0);

// D p with p = z r + a p formed on the way, for one system that is deferred or has one live shift
// (k_dslash_split_p): a.src holds p before the update, pnew takes it after the update, part the npart
// partial sums of |r|^2; x, if not deferred, takes x - beta p. Does nothing unless st->run is set. Only
// for one system on a lattice whose split term has 8 waves; refuses others.
template <typename S> struct CgmState;
template <class LF, class LL, typename SR>
void launch_dslash_p(DslashArgs<LF, LL, SR> a, CgmState<SR> *st, const c2_t<SR> *r, Vec<SR> pnew, Vec<SR> x,
                     const double *part, uint32_t npart, double *shist, hipStream_t stream);

// launch_dslash on vectors of the loaded gauge's precision in the caller's host layout (device memory,
// aligned to their reals): lay LAY_HOST with EPI_STORE (D src, nr right-hand sides per block), or
// the two terms of sigma0 src - D D src on one right-hand side, LAY_HOST_SRC with EPI_STORE and
// LAY_HOST_DST with EPI_AXMY, whose intermediate is in colour planes; or, in FP64, LAY_HOST_DST with
// EPI_STORE in blocks of 3, 4 or 8 (host_planes_block). The vectors of one launch
// must not overlap, except that aux and dst may be the same vector.
template <class LF, class LL, typename SR>
void launch_dslash_host(const DslashArgs<LF, LL, SR> &a, int lay, int epi, int nr, hipStream_t st);

// Block size for nrhs FP64 vectors in the host layout, of which the caller wants blocks of nr, if their
// source is first converted to colour planes, or 0 if the split term reads it as it is, in blocks of 2.
// Blocks of 3 and more would spill in the split form; with one thread per site they read the links
// less often, which pays above the sizes that the split term is for. Calls in blocks of 2 -> this,
// nr = 4 (nr = 8): 16^3x32 8 vectors 139 -> 113 us (104); 24^4 3 vectors 169 -> 124, 5 250 -> 218
// (173), 8 342 -> 256 (247); 32^4 3 500 -> 326, 5 750 -> 600 (422), 8 1027 -> 704 (678); 48^4 8
// 5450 -> 3521 (3353). Reading the host layout in blocks of 8 as well, without the conversion: 32^4 1287,
// 48^4 6307. The block is the one of least weight over all vectors: 29, 33 and 55 per block of 3, 4 and 8
// pick the faster one for 3 to 12 vectors at these sizes (padding costs less than its slots, since it
// repeats a vector).
inline int host_planes_block(const Geom &g, int nrhs, int nr)
{
    if (nr < 3 || nrhs < 3 || g.Vh <= kSplitSites64)
        return 0;
    const int c3 = (nrhs + 2) / 3 * 29, c4 = (nrhs + 3) / 4 * 33, c8 = (nrhs + 7) / 8 * 55;
    if (nr == 8 && c8 < c3 && c8 < c4)
        return 8;
    return c3 < c4 ? 3 : 4;
}

// Workgroups of nt sites for Vh sites, rounded up to a multiple of the 8 XCDs so that tile_site can
// give each XCD a contiguous range of sites on any lattice (the last ones may be empty)
inline uint32_t dslash_grid(uint32_t Vh, int nt)
{
    return (uint32_t)(((uint64_t)Vh + 8u * (uint32_t)nt - 1) / (8u * (uint32_t)nt)) * 8u;
}

inline uint32_t dslash_nblk(uint32_t Vh, int nt) { return dslash_grid(Vh, nt); }

// Row length Lx/2 of the lattices whose batched hopping terms stage rows in LDS (Lx = 32, as at
// 32^4): a compile-time row length gives the staged kernel a static LDS size
constexpr int kStageLxh = 16;

// KQ_STAGE=0 turns the LDS row staging of the batched hopping terms off (a tuning switch;
// results are bitwise the same either way)
inline bool stage_enabled()
{
    static const bool on = [] {
        const char *e = getenv("KQ_STAGE");
        return !(e && e[0] == '0');
    }();
    return on;
}

// Lattices whose workgroups of 256 cover whole x-rows of one (x, y) plane of that row length
inline bool stage_lattice(const Geom &g) { return g.lxh == kStageLxh && stage_rows(g, 256) > 0; }

// Whether launch_dslash runs the LDS-staged kernel for nr right-hand sides per thread and block
// size nt on this lattice (its NR * 3 * 352 staged colour entries, at most 67.6 KB for eight
// FP32 or 33.8 KB for two FP64 right-hand sides, fit a workgroup's LDS on gfx950)
inline bool dslash_staged(const Geom &g, int nr, int nt)
{
    return nr >= 2 && nt == 256 && stage_enabled() && stage_lattice(g);
}

// Waves per 64 sites of the split hopping term (k_dslash_split) that launch_dslash uses for nrhs
// right-hand sides in blocks of nr, or 0 where one thread per site serves better: when the
// one-thread form's waves (Vh / 64 per block) already fill the chip. Measured per term, one
// thread per site -> split: FP64 (blocks of 1) 8^4 8.9 -> 4.5 us, 16^4 18.9 -> 12.7, 22x18x15x13
// 20.6 -> 17.1, 16^3x32 23.9 -> 25.2; FP32 (LinkF, LinkF12) blocks of 1: 16^4 12.1 -> 7.1, 16^3x32
// 14.5 -> 12.6, 20^4 19.0 -> 16.4, 24^4 29.8 -> 31.2; blocks of 4: 16^4 21.8 -> 12.4, 16^3x32
// 23.8 -> 21.1, but two groups of 4 there 33 -> 37, 24^4 50 -> 47 (47.6 in workgroups of 64).
// Blocks of 8 FP32 right-hand sides leave the one-thread form one wave per SIMD, waiting for its
// gathers: split into 4 waves (or 2, hop_kernel) at every size, 16^4 41 -> 18, 24^4 82 -> 75, 48^4
// 1316 -> 1118, except where the larger lattices stage rows in LDS (32^4: 174 staged, 203 split).
//
// The two forms add the 16 hops in different orders. The FP64 rule therefore counts blocks of 2
// whatever nr is: nr comes from timings in the FP64 solve of several systems and in the FP64
// verification, whose results are the same in every process (repro_nt). Two or more FP64 vectors
// run faster as pairs on either form (two vectors in single blocks -> a pair: 16^4 20.7 -> 13.1 us, 24^4
// 115 -> 65, 32^4 354 -> 193, 48^4 1948 -> 1077; only at 8^4 4.4 -> 5.0), so the rule follows those.
inline int dslash_split_waves(bool fp64, const Geom &g, int nrhs, int nr)
{
    if (fp64)
        return nr <= 2 && (uint64_t)g.Vh * (uint64_t)((nrhs + 1) / 2) <= kSplitSites64 ? 8 : 0;
    if ((uint64_t)g.Vh * (uint64_t)((nrhs + nr - 1) / nr) <= kSplitSites32)
        return nr <= 2 ? 8 : 4;
    return nr == 8 && !stage_lattice(g) ? 4 : 0;
}

// The kernel of one hopping term on colour planes: waves per 64 sites of the split one (8, 4 or 2),
// kHopStaged for the one with rows in LDS, kHopSingle for one thread per site. small_long: long links
// of fewer than 40 bytes (LinkH12, LinkH12C). Their blocks of 8 on more than 48 K sites take 2 waves of
// 8 hops, whose 12.7 KB of LDS let all workgroups of a middle-sized lattice run at once (16^3x32 35 us
// with 4 waves, 30 with 2; 24^4 74 and 73.5, 48^4 1093 and 1040; but 16^4 17.6 and 24); the general
// 16-bit links (LinkH, 40 bytes) keep 4, which is all that was measured for them.
constexpr int kHopSingle = 0, kHopStaged = 1;
inline int hop_kernel(bool fp64, bool small_long, const Geom &g, int nrhs, int nr, int nt)
{
    const int waves = dslash_split_waves(fp64, g, nrhs, nr);
    if (waves > 0)
        return waves == 4 && nr == 8 && small_long && g.Vh > 49152u ? 2 : waves;
    return dslash_staged(g, nr, nt) ? kHopStaged : kHopSingle;
}

}  // namespace kq
