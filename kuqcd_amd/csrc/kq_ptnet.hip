// HIP kernels of the parallel-transport convolution preconditioner: the two
// forward layers (the second with an optional fused dot product for the
// flexible CG), the backward pass to the hidden layer, the weight gradients
// (deterministic two-stage FP64 reductions), and FP32 vector helpers.
#include <cstring>
#include <stdexcept>

#include "kq_ptnet.h"
#include "kq_solver.h"

namespace kq {

namespace {

constexpr int kNT = 256;  // threads per block of every kernel here

__device__ __forceinline__ float2 cmulf(float2 a, float2 b)
{
    return mk<float2>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__device__ __forceinline__ float2 unpack_w(uint32_t u)
{
    return mk<float2>(__uint_as_float(u << 16), __uint_as_float(u & 0xffff0000u));
}

// (re, im) -> bfloat16 pair in unpack_w's format, round to nearest even (finite values)
__device__ __forceinline__ uint32_t pack_bf16(float2 v)
{
    uint32_t a = __float_as_uint(v.x), b = __float_as_uint(v.y);
    a += 0x7fffu + ((a >> 16) & 1u);
    b += 0x7fffu + ((b >> 16) & 1u);
    return (a >> 16) | (b & 0xffff0000u);
}

// Neighbours of (s, coordinates) along the direction mu of a wave, a value uniform over the wave: hops
// +1, +3, -1, -3 (the taps t = 4 mu + 0..3). The direction stays a run-time value, with its
// coordinate, extent and weights selected: specialised code for each wave's direction behind
// branches on the wave index was compiled wrongly (one wave took other taps' weights, and with
// 16-bit links an address that was never set).
struct DirNb {
    uint32_t n[4];
};
__device__ __forceinline__ DirNb dir_neighbours(const Geom &g, uint32_t s, const SiteCoord &sc, int mu)
{
    const int c = mu == 0 ? sc.c[0] : mu == 1 ? sc.c[1] : mu == 2 ? sc.c[2] : sc.c[3];
    const int L = g.L[mu];
    const uint32_t stride = g.stride[mu];
    const int h[4] = {1, 3, -1, -3};
    DirNb d;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int v = wrap_add(c, h[t], L);
        d.n[t] = s + (mu == 0 ? (uint32_t)((v >> 1) - (c >> 1)) : (uint32_t)(v - c) * stride);
    }
    return d;
}

// The kernel's first argument in the argument segment: values indexed by the direction come from there
// by scalar loads (indexing the by-value argument itself would copy it to scratch memory)
template <class T> __device__ __forceinline__ const T &first_arg()
{
    return *(const T *)__builtin_amdgcn_kernarg_segment_ptr();
}
template <class F> struct FirstParam;
template <class T, class... R> struct FirstParam<void (*)(T, R...)> {
    using type = T;
};
// to stand beside each kernel that calls first_arg<T>(): T is its first parameter
#define KQ_FIRST_ARG(T, ...) \
    static_assert(std::is_same<FirstParam<decltype(&__VA_ARGS__)>::type, T>::value, "first_arg reads the first parameter")

// The links of the four taps: every load is issued before any is used
template <class LF, class LL>
__device__ __forceinline__ void dir_links(const LF &fat, const LL &lng, int qo, int mu, uint32_t s, const DirNb &d,
                                          float2 U[4][9])
{
    fat.load(qo, mu, s, U[0]);
    lng.load(qo, mu, s, U[1]);
    fat.load(1 - qo, mu, d.n[2], U[2]);
    lng.load(1 - qo, mu, d.n[3], U[3]);
}

// v = U x for a forward tap (t < 2), U^+ x for a backward one
__device__ __forceinline__ void tap_mul(int t, const float2 U[9], const float2 x[3], float2 v[3])
{
    float acc[6] = {0, 0, 0, 0, 0, 0};
    if (t < 2) {
        umv_add(U, x, acc);
    } else {
        udmv_sub(U, x, acc);
#pragma unroll
        for (int k = 0; k < 6; ++k)
            acc[k] = -acc[k];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k)
        v[k] = mk<float2>(acc[2 * k], acc[2 * k + 1]);
}

// (T_t in)(s) for a one-channel field `in` on parity 1-qo, the four taps of direction mu
template <class LF, class LL>
__device__ __forceinline__ void taps1_dir(const Geom &g, int qo, const LF &fat, const LL &lng, uint32_t s, int mu,
                                          const float2 *in, float2 v[4][3])
{
    const DirNb d = dir_neighbours(g, s, site_coords(g, s, qo), mu);
    float2 x[4][3], U[4][9];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int c = 0; c < 3; ++c)
            x[t][c] = in[(size_t)c * g.Vh + d.n[t]];
    dir_links(fat, lng, qo, mu, s, d, U);
#pragma unroll
    for (int t = 0; t < 4; ++t)
        tap_mul(t, U[t], x[t], v[t]);
}

// The layers and the weight gradient give the 64 sites of a workgroup to 4 waves, one per direction
// (4 of the 16 taps each), as k_dslash_split does with its hops: 4 times the waves in flight and a
// quarter of the chain of dependent loads of one thread per site, and workgroups of 64 sites end a
// grid evenly. One thread per site in workgroups of 256 -> 4 waves per 64 sites: see the kernels.
constexpr int kSites = 64;

struct PtLayerArgs {
    Geom g;
    int qo;              // output parity
    const float2 *in;    // input field(s) on parity 1-qo, channel stride 3*Vh
    float2 *out;         // output field(s) on parity qo, channel stride 3*Vh (may be null with out16)
    kq_v4u *out16;       // layer 1: the outputs also as bfloat16 (pt_forward's h16 layout); may be null
    const kq_v4u *in16;  // layer 2: read the channels from here (bfloat16) instead of in; may be null
    const float2 *skip;  // layer 2: w0 * skip(x) added (parity qo); may be null
    const float2 *dotq;  // layer 2: per-block partials of <dotq, out> (may be null)
    double *part;        // [2*nblk]
    const int *stop;     // do nothing while *stop != 0 (may be null)
    PtWeightsBF w;       // layer-1 form uses w1; layer-2 form uses w2 and w0
};

// acc[c][k] += sum over direction mu's taps of w1[c][t] (T_t in)_k
template <class LF, class LL>
__device__ __forceinline__ void layer1_dir(const PtLayerArgs &a, const LF &fat, const LL &lng, uint32_t s, int mu,
                                           float2 acc[kPtHidden][3])
{
    float2 v[4][3];
    taps1_dir(a.g, a.qo, fat, lng, s, mu, a.in, v);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int c = 0; c < kPtHidden; ++c) {
            const float2 w = unpack_w(a.w.w1[c][4 * mu + t]);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const float2 p = cmulf(w, v[t][k]);
                acc[c][k].x += p.x;
                acc[c][k].y += p.y;
            }
        }
}

// layer-1 form: out_c(x) = sum_t w1[c][t] (T_t in)(x), one input channel, kPtHidden outputs
template <class LF, class LL>
__global__ void __launch_bounds__(kNT) k_pt_layer1(const PtLayerArgs a, LF fat, LL lng)
{
    static_assert(kNT == 4 * kSites, "one wave per direction");
    constexpr int NV = 2 * 3 * kPtHidden;
    __shared__ float red[2][NV][kSites];
    __shared__ uint32_t site[kSites];
    if (a.stop && *a.stop)
        return;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    bool valid;
    const uint32_t s = tile_site<kSites>(a.g, blockIdx.x, gridDim.x, lane, valid);
    float2 acc[kPtHidden][3];
#pragma unroll
    for (int c = 0; c < kPtHidden; ++c)
#pragma unroll
        for (int k = 0; k < 3; ++k)
            acc[c][k] = mk<float2>(0.f, 0.f);
    if (valid)
        layer1_dir(first_arg<PtLayerArgs>(), fat, lng, s, w, acc);
    if (w == 0)
        site[lane] = valid ? s : 0xffffffffu;
    if (w >= 2) {
#pragma unroll
        for (int c = 0; c < kPtHidden; ++c)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                red[w - 2][6 * c + 2 * k][lane] = acc[c][k].x;
                red[w - 2][6 * c + 2 * k + 1][lane] = acc[c][k].y;
            }
    }
    __syncthreads();
    if (w < 2) {
#pragma unroll
        for (int c = 0; c < kPtHidden; ++c)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                red[w][6 * c + 2 * k][lane] += acc[c][k].x;
                red[w][6 * c + 2 * k + 1][lane] += acc[c][k].y;
            }
    }
    __syncthreads();
    const uint32_t sl = site[lane];
    if (sl == 0xffffffffu)
        return;
    const auto entry = [&](int c, int k) {
        return mk<float2>(red[0][6 * c + 2 * k][lane] + red[1][6 * c + 2 * k][lane],
                          red[0][6 * c + 2 * k + 1][lane] + red[1][6 * c + 2 * k + 1][lane]);
    };
    if (a.out) {  // wave w writes channel w
        static_assert(kPtHidden == 4, "one wave per channel");
#pragma unroll
        for (int k = 0; k < 3; ++k)
            a.out[((size_t)w * 3 + k) * a.g.Vh + sl] = entry(w, k);
    }
    if (a.out16 && w < 3) {  // wave w writes colour w
        static_assert(kPtHidden == 4, "the bfloat16 hidden layout holds 4 channels");
        kq_v4u u;
        u.x = pack_bf16(entry(0, w));
        u.y = pack_bf16(entry(1, w));
        u.z = pack_bf16(entry(2, w));
        u.w = pack_bf16(entry(3, w));
        a.out16[(size_t)w * a.g.Vh + sl] = u;
    }
}
KQ_FIRST_ARG(PtLayerArgs, k_pt_layer1<LinkF, LinkF>);

// acc += sum over direction mu's taps of T_t( sum_c w2[c][t] in_c ). With bfloat16 channels one
// 16-byte load brings the four channels of one colour, and the 12 gathers and the link loads are all
// issued before any is used (written tap by tap the compiler waited for each 16-byte gather).
template <class LF, class LL, bool H16>
__device__ __forceinline__ void layer2_dir(const PtLayerArgs &a, const LF &fat, const LL &lng, uint32_t s, int mu,
                                           float2 acc[3])
{
    const uint32_t Vh = a.g.Vh;
    const DirNb d = dir_neighbours(a.g, s, site_coords(a.g, s, a.qo), mu);
    float2 x[4][3], U[4][9];
    kq_v4u u[4][3];
    if constexpr (H16) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int c = 0; c < 3; ++c)
                u[t][c] = a.in16[(size_t)c * Vh + d.n[t]];
        dir_links(fat, lng, a.qo, mu, s, d, U);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        float2 wt[kPtHidden];
#pragma unroll
        for (int ch = 0; ch < kPtHidden; ++ch)
            wt[ch] = unpack_w(a.w.w2[ch][4 * mu + t]);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            if constexpr (H16) {
                const float2 p0 = cmulf(wt[0], unpack_w(u[t][c].x)), p1 = cmulf(wt[1], unpack_w(u[t][c].y));
                const float2 p2 = cmulf(wt[2], unpack_w(u[t][c].z)), p3 = cmulf(wt[3], unpack_w(u[t][c].w));
                x[t][c] = mk<float2>((p0.x + p1.x) + (p2.x + p3.x), (p0.y + p1.y) + (p2.y + p3.y));
            } else {
                x[t][c] = mk<float2>(0.f, 0.f);
#pragma unroll
                for (int ch = 0; ch < kPtHidden; ++ch) {
                    const float2 p = cmulf(wt[ch], a.in[((size_t)ch * 3 + c) * Vh + d.n[t]]);
                    x[t][c].x += p.x;
                    x[t][c].y += p.y;
                }
            }
        }
    }
    if constexpr (!H16)
        dir_links(fat, lng, a.qo, mu, s, d, U);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        float2 v[3];
        tap_mul(t, U[t], x[t], v);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            acc[k].x += v[k].x;
            acc[k].y += v[k].y;
        }
    }
}

// layer-2 form: out(x) = w0 skip(x) + sum_t T_t( sum_c w2[c][t] in_c )(x); H16: channels from in16
template <class LF, class LL, bool H16>
__global__ void __launch_bounds__(kNT) __attribute__((amdgpu_waves_per_eu(1, 4)))
k_pt_layer2(const PtLayerArgs a, LF fat, LL lng)
{
    __shared__ float red[4][6][kSites];
    __shared__ double lre[kNT / kWave], lim[kNT / kWave];
    if (a.stop && *a.stop)
        return;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    bool valid;
    const uint32_t s = tile_site<kSites>(a.g, blockIdx.x, gridDim.x, lane, valid);
    float2 acc[3] = {mk<float2>(0.f, 0.f), mk<float2>(0.f, 0.f), mk<float2>(0.f, 0.f)};
    if (valid)
        layer2_dir<LF, LL, H16>(first_arg<PtLayerArgs>(), fat, lng, s, w, acc);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        red[w][2 * k][lane] = acc[k].x;
        red[w][2 * k + 1][lane] = acc[k].y;
    }
    __syncthreads();
    // wave k < 3 finishes colour k
    double re = 0.0, im = 0.0;
    if (w < 3 && valid) {
        const size_t e = (size_t)w * a.g.Vh + s;
        float2 z = a.skip ? cmulf(unpack_w(a.w.w0), a.skip[e]) : mk<float2>(0.f, 0.f);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            z.x += red[d][2 * w][lane];
            z.y += red[d][2 * w + 1][lane];
        }
        a.out[e] = z;
        if (a.dotq) {
            const float2 d = a.dotq[e];
            re = (double)d.x * z.x + (double)d.y * z.y;
            im = (double)d.x * z.y - (double)d.y * z.x;
        }
    }
    if (a.dotq) {
        re = wave_sum(re);
        im = wave_sum(im);
        if (lane == 0) {
            lre[w] = re;
            lim[w] = im;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            a.part[2 * blockIdx.x] = (lre[0] + lre[1]) + lre[2];
            a.part[2 * blockIdx.x + 1] = (lim[0] + lim[1]) + lim[2];
        }
    }
}
KQ_FIRST_ARG(PtLayerArgs, k_pt_layer2<LinkF, LinkF, true>);

// P[c][t] = sum over sites y of parity qo of <(T_t in)(y), b_c(y)> for the two (in, b) pairs of a
// gradient (blockIdx.y); part[pair][blk][c*16 + t] (complex, FP64).
// Each wave forms the four tap vectors of its direction for the workgroup's 64 sites in LDS; then
// every thread owns one (c, t) and a quarter of the sites and adds the FP64 products over them.
// (Before, each thread kept its site and every one of the 64 complex sums was reduced over the
// wave by 12 shuffles, 1536 in all: 41 us a pair at 16^4.) The strides of 98 and 26 floats put the
// 64 threads of a wave on distinct banks in both phases.
struct PtGradArgs {
    const float2 *in[2], *b[2];
};

constexpr int kTapStride = 6 * kPtTaps + 2, kChanStride = 6 * kPtHidden + 2;

template <class LF, class LL>
__global__ void __launch_bounds__(kNT) k_pt_wgrad(Geom g, int qo, LF fat, LL lng, const PtGradArgs p, double2 *part)
{
    constexpr int J = kJ;
    static_assert(J == kWave && kPtHidden == kNT / kWave, "one (c, t) per lane, one channel per wave");
    __shared__ __align__(8) float tv[kSites * kTapStride];
    __shared__ __align__(8) float bv[kSites * kChanStride];
    __shared__ double2 sum[kNT / kWave][J];
    const float2 *in = p.in[blockIdx.y], *b = p.b[blockIdx.y];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    bool valid;
    const uint32_t s = tile_site<kSites>(g, blockIdx.x, gridDim.x, lane, valid);
    float2 *row = reinterpret_cast<float2 *>(tv + lane * kTapStride);
    if (valid) {
        float2 v[4][3];
        taps1_dir(first_arg<Geom>(), qo, fat, lng, s, w, in, v);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int k = 0; k < 3; ++k)
                row[12 * w + 3 * t + k] = v[t][k];
    } else {
#pragma unroll
        for (int k = 0; k < 12; ++k)
            row[12 * w + k] = mk<float2>(0.f, 0.f);
    }
#pragma unroll
    for (int k = 0; k < 3; ++k)
        reinterpret_cast<float2 *>(bv + lane * kChanStride)[3 * w + k] =
            valid ? b[((size_t)w * 3 + k) * g.Vh + s] : mk<float2>(0.f, 0.f);
    __syncthreads();
    const int t = lane & (kPtTaps - 1), c = lane / kPtTaps;
    double re = 0.0, im = 0.0;
    for (int i = w * (kSites / 4); i < (w + 1) * (kSites / 4); ++i) {
        const float2 *v = reinterpret_cast<const float2 *>(tv + i * kTapStride) + 3 * t;
        const float2 *bb = reinterpret_cast<const float2 *>(bv + i * kChanStride) + 3 * c;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double vx = v[k].x, vy = v[k].y, bx = bb[k].x, by = bb[k].y;
            re = fmadd(vx, bx, re);
            re = fmadd(vy, by, re);
            im = fmadd(vx, by, im);
            im = fmadd(-vy, bx, im);
        }
    }
    sum[w][lane] = mk<double2>(re, im);
    __syncthreads();
    if (w == 0) {
        double2 o = sum[0][lane];
#pragma unroll
        for (int k = 1; k < kNT / kWave; ++k) {
            o.x += sum[k][lane].x;
            o.y += sum[k][lane].y;
        }
        part[((size_t)blockIdx.y * gridDim.x + blockIdx.x) * J + lane] = o;
    }
}
KQ_FIRST_ARG(Geom, k_pt_wgrad<LinkF, LinkF>);

// out[y*gridDim.x + j] = sum over blocks b of part[(y*nblk + b)*stride + j], j = blockIdx.x,
// y = blockIdx.y < 2; fixed summation order. For y = 2, j < 2: the sums over the nblk2 entries of
// part2 + j*nblk2.
__global__ void __launch_bounds__(kNT) k_reduce_cols(const double2 *part, uint32_t nblk, uint32_t stride,
                                                     double2 *out, const double2 *part2, uint32_t nblk2)
{
    int j = blockIdx.x;
    out += (size_t)blockIdx.y * gridDim.x + j;
    if (blockIdx.y == 2) {
        if (j > 1)
            return;
        part = part2 + (size_t)j * nblk2;
        nblk = nblk2;
        stride = 1;
        j = 0;
    } else {
        part += (size_t)blockIdx.y * nblk * stride;
    }
    __shared__ double lre[kNT], lim[kNT];
    double re = 0.0, im = 0.0;
    for (uint32_t b = threadIdx.x; b < nblk; b += kNT) {
        const double2 v = part[(size_t)b * stride + j];
        re += v.x;
        im += v.y;
    }
    lre[threadIdx.x] = re;
    lim[threadIdx.x] = im;
    __syncthreads();
    for (int w = kNT / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            lre[threadIdx.x] += lre[threadIdx.x + w];
            lim[threadIdx.x] += lim[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        *out = mk<double2>(lre[0], lim[0]);
}

__global__ void k_vf_lincomb(float2 *y, const float2 *x1, float2 a1, const float2 *x2, float2 a2, size_t n)
{
    const size_t i = (size_t)blockIdx.x * kNT + threadIdx.x;
    if (i < n) {
        const float2 p = cmulf(a1, x1[i]), q = cmulf(a2, x2[i]);
        y[i] = mk<float2>(p.x + q.x, p.y + q.y);
    }
}

struct DotSet {
    const float2 *x[8];
    const float2 *y[8];
};

// part[k*nblk + blk] = block partial of <x_k, y_k>
__global__ void __launch_bounds__(kNT) k_vf_dots(DotSet d, int nd, size_t n, double2 *part)
{
    __shared__ double lre[kNT / kWave], lim[kNT / kWave];
    const size_t i = (size_t)blockIdx.x * kNT + threadIdx.x;
    for (int k = 0; k < nd; ++k) {
        double re = 0.0, im = 0.0;
        if (i < n) {
            const float2 a = d.x[k][i], b = d.y[k][i];
            re = (double)a.x * b.x + (double)a.y * b.y;
            im = (double)a.x * b.y - (double)a.y * b.x;
        }
        re = wave_sum(re);
        im = wave_sum(im);
        if ((threadIdx.x & (kWave - 1)) == 0) {
            lre[threadIdx.x / kWave] = re;
            lim[threadIdx.x / kWave] = im;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double sr = 0.0, si = 0.0;
            for (int w = 0; w < kNT / kWave; ++w) {
                sr += lre[w];
                si += lim[w];
            }
            part[(size_t)k * gridDim.x + blockIdx.x] = mk<double2>(sr, si);
        }
        __syncthreads();
    }
}

struct SumsqSet {
    const double *x[2];
    size_t n[2];
    uint32_t nb[2];
};

// part[y*kSumsqParts + blk] = block partial of |x_y|^2, y = blockIdx.y
__global__ void __launch_bounds__(kNT) k_vd_sumsq(SumsqSet a, double *part)
{
    __shared__ double l[kNT / kWave];
    const int y = blockIdx.y;
    const double *x = a.x[y];
    const uint32_t nb = a.nb[y];
    if (blockIdx.x >= nb)
        return;
    double acc = 0.0;
    for (size_t i = (size_t)blockIdx.x * kNT + threadIdx.x; i < a.n[y]; i += (size_t)nb * kNT)
        acc += x[i] * x[i];
    acc = wave_sum(acc);
    if ((threadIdx.x & (kWave - 1)) == 0)
        l[threadIdx.x / kWave] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int w = 0; w < kNT / kWave; ++w)
            s += l[w];
        part[(size_t)y * kSumsqParts + blockIdx.x] = s;
    }
}

__global__ void k_vd_set(double *p, double v) { *p = v; }

// block sum of (a, b), valid in thread 0
__device__ __forceinline__ double2 block_sum2(double a, double b)
{
    __shared__ double la[kNT / kWave], lb[kNT / kWave];
    a = wave_sum(a);
    b = wave_sum(b);
    if ((threadIdx.x & (kWave - 1)) == 0) {
        la[threadIdx.x / kWave] = a;
        lb[threadIdx.x / kWave] = b;
    }
    __syncthreads();
    double2 o = mk<double2>(0.0, 0.0);
    for (int w = 0; w < kNT / kWave; ++w) {
        o.x += la[w];
        o.y += lb[w];
    }
    return o;
}

// d = az - ae; part[blk] = (|d|^2, |ae|^2)
__global__ void __launch_bounds__(kNT) k_loss_residual(const float2 *az, const float2 *ae, float2 *d, size_t n,
                                                       double2 *part)
{
    double dd = 0.0, aa = 0.0;
    for (size_t i = (size_t)blockIdx.x * kNT + threadIdx.x; i < n; i += (size_t)gridDim.x * kNT) {
        const float2 p = az[i], q = ae[i], o = mk<float2>(p.x - q.x, p.y - q.y);
        d[i] = o;
        dd += (double)o.x * o.x + (double)o.y * o.y;
        aa += (double)q.x * q.x + (double)q.y * q.y;
    }
    const double2 t = block_sum2(dd, aa);
    if (threadIdx.x == 0)
        part[blockIdx.x] = t;
}

// g = g / |ae|^2 with |ae|^2 the sum over the nblk partials of k_loss_residual, added here by every
// block in the same order; part[blk] = <r, g>. The host sees |ae|^2 after the gradient and drops
// the gradient if it is not positive.
__global__ void __launch_bounds__(kNT) k_loss_scale(const double2 *part_loss, uint32_t nblk, float2 *g,
                                                    const float2 *r, size_t n, double2 *part)
{
    __shared__ double l[kNT / kWave];
    double den = 0.0;
    for (uint32_t k = threadIdx.x; k < nblk; k += kNT)
        den += part_loss[k].y;
    den = wave_sum(den);
    if ((threadIdx.x & (kWave - 1)) == 0)
        l[threadIdx.x / kWave] = den;
    __syncthreads();
    den = (l[0] + l[1]) + (l[2] + l[3]);
    const float inv = den > 0.0 ? (float)(1.0 / den) : 0.f;
    double re = 0.0, im = 0.0;
    for (size_t i = (size_t)blockIdx.x * kNT + threadIdx.x; i < n; i += (size_t)gridDim.x * kNT) {
        const float2 o = mk<float2>(inv * g[i].x, inv * g[i].y), a = r[i];
        g[i] = o;
        re += (double)a.x * o.x + (double)a.y * o.y;
        im += (double)a.x * o.y - (double)a.y * o.x;
    }
    const double2 t = block_sum2(re, im);
    if (threadIdx.x == 0)
        part[blockIdx.x] = t;
}

__global__ void __launch_bounds__(kNT) k_unpack_hidden(const kq_v4u *h16, float2 *h, uint32_t Vh)
{
    const size_t i = (size_t)blockIdx.x * kNT + threadIdx.x;  // colour-major entry k*Vh + s
    if (i >= (size_t)3 * Vh)
        return;
    const kq_v4u u = h16[i];
    const size_t n3 = (size_t)3 * Vh;
    h[i] = unpack_w(u.x);
    h[n3 + i] = unpack_w(u.y);
    h[2 * n3 + i] = unpack_w(u.z);
    h[3 * n3 + i] = unpack_w(u.w);
}

inline unsigned grid_of(size_t n) { return (unsigned)((n + kNT - 1) / kNT); }

}  // namespace

void pt_unpack_hidden(const kq_v4u *h16, float2 *h, uint32_t Vh, hipStream_t st)
{
    if (Vh == 0)
        return;
    hipLaunchKernelGGL(k_unpack_hidden, dim3(grid_of((size_t)3 * Vh)), dim3(kNT), 0, st, h16, h, Vh);
    KQ_HIP_CHECK(hipGetLastError());
}

uint32_t pt_layer_nblk(uint32_t Vh) { return dslash_grid(Vh, kSites); }

template <class LF, class LL>
void pt_forward(const Geom &g, int q, LF fat, LL lng, const PtWeightsBF &w, const float2 *r, float2 *h, float2 *z,
                hipStream_t st, const float2 *dotq, double *part, const int *stop, kq_v4u *h16)
{
    if (g.Vh == 0)
        return;
    const unsigned nb = pt_layer_nblk(g.Vh);
    PtLayerArgs a{};
    a.g = g;
    a.w = w;
    a.stop = stop;
    a.qo = 1 - q;
    a.in = r;
    a.out = h;
    a.out16 = h16;
    hipLaunchKernelGGL((k_pt_layer1<LF, LL>), dim3(nb), dim3(kNT), 0, st, a, fat, lng);
    KQ_HIP_CHECK(hipGetLastError());
    a.qo = q;
    a.in = h;
    a.in16 = h16;
    a.out16 = nullptr;
    a.out = z;
    a.skip = r;
    a.dotq = dotq;
    a.part = part;
    if (h16)
        hipLaunchKernelGGL((k_pt_layer2<LF, LL, true>), dim3(nb), dim3(kNT), 0, st, a, fat, lng);
    else
        hipLaunchKernelGGL((k_pt_layer2<LF, LL, false>), dim3(nb), dim3(kNT), 0, st, a, fat, lng);
    KQ_HIP_CHECK(hipGetLastError());
}

template <class LF, class LL>
void pt_backward_hidden(const Geom &g, int q, LF fat, LL lng, const PtWeightsBF &wb, const float2 *gz, float2 *gh,
                        hipStream_t st)
{
    if (g.Vh == 0)
        return;
    PtLayerArgs a{};
    a.g = g;
    a.w = wb;
    a.qo = 1 - q;
    a.in = gz;
    a.out = gh;
    hipLaunchKernelGGL((k_pt_layer1<LF, LL>), dim3(pt_layer_nblk(g.Vh)), dim3(kNT), 0, st, a, fat, lng);
    KQ_HIP_CHECK(hipGetLastError());
}

template <class LF, class LL>
void pt_weight_grads(const Geom &g, int q, LF fat, LL lng, const float2 *r, const float2 *h, const float2 *gz,
                     const float2 *gh, double2 *part, hipStream_t st)
{
    if (g.Vh == 0)
        return;
    // gW1[c][t] = sum_y <T_t r, gh_c>, y on parity 1-q
    // gW2[c][t] = sum_y <h_c, T_{flip t} g> = conj(sum_y <T_{flip t} g, h_c>)
    const PtGradArgs p{{r, gz}, {gh, h}};
    hipLaunchKernelGGL((k_pt_wgrad<LF, LL>), dim3(pt_layer_nblk(g.Vh), 2), dim3(kNT), 0, st, g, 1 - q, fat, lng, p,
                       part);
    KQ_HIP_CHECK(hipGetLastError());
}

size_t pt_grad_parts(uint32_t Vh) { return (size_t)pt_layer_nblk(Vh) * 2 * kJ; }

void pt_reduce(const double2 *grad_part, const double2 *loss_part, uint32_t Vh, size_t n, double2 *out,
               hipStream_t st)
{
    hipLaunchKernelGGL(k_reduce_cols, dim3(kJ, 3), dim3(kNT), 0, st, grad_part, grad_part ? pt_layer_nblk(Vh) : 0u,
                       (uint32_t)kJ, out, loss_part, loss_nblk(n));
    KQ_HIP_CHECK(hipGetLastError());
}

void pt_unpack_grads(const double2 *sums, double *out)
{
    for (int c = 0; c < kPtHidden; ++c)
        for (int t = 0; t < kPtTaps; ++t) {
            const int j1 = c * kPtTaps + t, j2 = kJ + c * kPtTaps + t;
            out[2 * j1] = sums[j1].x;
            out[2 * j1 + 1] = sums[j1].y;
            const double2 b = sums[kJ + c * kPtTaps + pt_flip_tap(t)];
            out[2 * j2] = b.x;
            out[2 * j2 + 1] = -b.y;
        }
    // gW0 = sum_x <r, g>
    out[4 * kJ] = sums[kPtSumRG].x;
    out[4 * kJ + 1] = sums[kPtSumRG].y;
}

uint32_t loss_nblk(size_t n) { return (uint32_t)std::min<size_t>(512, grid_of(n)); }

void loss_residual(const float2 *az, const float2 *ae, float2 *d, size_t n, double2 *part, hipStream_t st)
{
    hipLaunchKernelGGL(k_loss_residual, dim3(loss_nblk(n)), dim3(kNT), 0, st, az, ae, d, n, part);
    KQ_HIP_CHECK(hipGetLastError());
}

void loss_scale(const double2 *part_loss, float2 *g, const float2 *r, size_t n, double2 *part, hipStream_t st)
{
    hipLaunchKernelGGL(k_loss_scale, dim3(loss_nblk(n)), dim3(kNT), 0, st, part_loss, loss_nblk(n), g, r, n, part);
    KQ_HIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------- weights
float bf16_round(float f)
{
    uint32_t u;
    std::memcpy(&u, &f, 4);
    if ((u & 0x7f800000u) == 0x7f800000u)
        return f;  // inf / nan unchanged
    u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest, ties to even
    u &= 0xffff0000u;
    float r;
    std::memcpy(&r, &u, 4);
    return r;
}

uint32_t bf16_pack(float2 w)
{
    const float re = bf16_round(w.x), im = bf16_round(w.y);
    uint32_t ur, ui;
    std::memcpy(&ur, &re, 4);
    std::memcpy(&ui, &im, 4);
    return (ur >> 16) | (ui & 0xffff0000u);
}

float2 bf16_unpack(uint32_t u)
{
    const uint32_t ur = u << 16, ui = u & 0xffff0000u;
    float re, im;
    std::memcpy(&re, &ur, 4);
    std::memcpy(&im, &ui, 4);
    return mk<float2>(re, im);
}

static float2 scaled(float2 w, double s) { return mk<float2>((float)(w.x * s), (float)(w.y * s)); }

PtWeightsBF pt_pack(const PtWeights &w, const PtNorms &nu)
{
    PtWeightsBF o{};
    for (int c = 0; c < kPtHidden; ++c)
        for (int t = 0; t < kPtTaps; ++t) {
            const double s = 1.0 / nu.nu[pt_tap_hop(t) == 3 ? 1 : 0];
            o.w1[c][t] = bf16_pack(scaled(w.w1[c][t], s));
            o.w2[c][t] = bf16_pack(scaled(w.w2[c][t], s));
        }
    o.w0 = bf16_pack(w.w0);
    return o;
}

PtWeightsBF pt_pack_backward(const PtWeights &w, const PtNorms &nu)
{
    const PtWeights e = pt_effective(w, nu);
    PtWeightsBF o{};
    for (int c = 0; c < kPtHidden; ++c)
        for (int t = 0; t < kPtTaps; ++t) {
            const float2 v = e.w2[c][pt_flip_tap(t)];
            o.w1[c][t] = bf16_pack(mk<float2>(v.x, -v.y));  // exact: v is already bf16
        }
    return o;
}

PtWeights pt_effective(const PtWeights &w, const PtNorms &nu)
{
    const PtWeightsBF p = pt_pack(w, nu);
    PtWeights o{};
    for (int c = 0; c < kPtHidden; ++c)
        for (int t = 0; t < kPtTaps; ++t) {
            o.w1[c][t] = bf16_unpack(p.w1[c][t]);
            o.w2[c][t] = bf16_unpack(p.w2[c][t]);
        }
    o.w0 = bf16_unpack(p.w0);
    return o;
}

// ---------------------------------------------------------------- vector helpers
void vf_lincomb(float2 *y, const float2 *x1, float2 a1, const float2 *x2, float2 a2, size_t n, hipStream_t st)
{
    if (n == 0)
        return;
    hipLaunchKernelGGL(k_vf_lincomb, dim3(grid_of(n)), dim3(kNT), 0, st, y, x1, a1, x2, a2, n);
    KQ_HIP_CHECK(hipGetLastError());
}

void vf_dots(const float2 *const *xs, const float2 *const *ys, int ndot, size_t n, double2 *out, hipStream_t st)
{
    if (ndot <= 0 || ndot > 8)
        throw std::invalid_argument("vf_dots: 1..8 dot products per launch");
    if (n == 0) {
        for (int k = 0; k < ndot; ++k)
            out[k] = mk<double2>(0.0, 0.0);
        return;
    }
    DotSet d{};
    for (int k = 0; k < ndot; ++k) {
        d.x[k] = xs[k];
        d.y[k] = ys[k];
    }
    const unsigned nb = grid_of(n);
    DevBuf part(sizeof(double2) * ndot * nb), res(sizeof(double2) * ndot);
    hipLaunchKernelGGL(k_vf_dots, dim3(nb), dim3(kNT), 0, st, d, ndot, n, part.as<double2>());
    KQ_HIP_CHECK(hipGetLastError());
    for (int k = 0; k < ndot; ++k) {
        hipLaunchKernelGGL(k_reduce_cols, dim3(1), dim3(kNT), 0, st, part.as<double2>() + (size_t)k * nb, nb, 1u,
                           res.as<double2>() + k, nullptr, 0u);
        KQ_HIP_CHECK(hipGetLastError());
    }
    KQ_HIP_CHECK(hipMemcpyAsync(out, res.as<void>(), sizeof(double2) * ndot, hipMemcpyDeviceToHost, st));
    KQ_HIP_CHECK(hipStreamSynchronize(st));
}

static uint32_t sumsq_nblk(size_t n) { return (uint32_t)std::min<size_t>(kSumsqParts, grid_of(n)); }

void vd_sumsq_partials(const double *const *x, const size_t *n, int count, double *part, hipStream_t st)
{
    SumsqSet a{};
    uint32_t nb = 0;
    for (int y = 0; y < count; ++y) {
        a.x[y] = x[y];
        a.n[y] = n[y];
        a.nb[y] = sumsq_nblk(n[y]);
        nb = std::max(nb, a.nb[y]);
    }
    if (nb == 0)
        return;
    hipLaunchKernelGGL(k_vd_sumsq, dim3(nb, count), dim3(kNT), 0, st, a, part);
    KQ_HIP_CHECK(hipGetLastError());
}

double vd_sumsq_total(const double *part, size_t n)
{
    double s = 0.0;
    for (uint32_t k = 0; k < sumsq_nblk(n); ++k)
        s += part[k];
    return s;
}

void vd_set(double *p, double v, hipStream_t st)
{
    hipLaunchKernelGGL(k_vd_set, dim3(1), dim3(1), 0, st, p, v);
    KQ_HIP_CHECK(hipGetLastError());
}

double vd_sumsq(const double *x, size_t n, hipStream_t st)
{
    if (n == 0)
        return 0.0;
    DevBuf part(sizeof(double) * kSumsqParts);
    vd_sumsq_partials(&x, &n, 1, part.as<double>(), st);
    std::vector<double> h(sumsq_nblk(n));
    KQ_HIP_CHECK(hipMemcpyAsync(h.data(), part.as<void>(), sizeof(double) * h.size(), hipMemcpyDeviceToHost, st));
    KQ_HIP_CHECK(hipStreamSynchronize(st));
    return vd_sumsq_total(h.data(), n);
}

#define KQ_PT_INST(LF, LL)                                                                                          \
    template void pt_forward<LF, LL>(const Geom &, int, LF, LL, const PtWeightsBF &, const float2 *, float2 *,       \
                                     float2 *, hipStream_t, const float2 *, double *, const int *, kq_v4u *);       \
    template void pt_backward_hidden<LF, LL>(const Geom &, int, LF, LL, const PtWeightsBF &, const float2 *,         \
                                             float2 *, hipStream_t);                                                \
    template void pt_weight_grads<LF, LL>(const Geom &, int, LF, LL, const float2 *, const float2 *,                 \
                                          const float2 *, const float2 *, double2 *, hipStream_t);
KQ_PT_INST(LinkF, LinkF)
KQ_PT_INST(LinkF, LinkF12)
KQ_PT_INST(LinkH, LinkH12)
KQ_PT_INST(LinkH, LinkH)
KQ_PT_INST(LinkF, LinkH12)
KQ_PT_INST(LinkF, LinkH)
KQ_PT_INST(LinkF, LinkF12C)
KQ_PT_INST(LinkH, LinkH12C)
KQ_PT_INST(LinkF, LinkH12C)

}  // namespace kq
