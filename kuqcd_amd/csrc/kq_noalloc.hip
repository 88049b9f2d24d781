// kq_mdaggm_noalloc: dst = sigma src - D D src (the CGM operator A, as kq_mdaggm)
// for callers that cannot allocate device memory (code under HIP graph capture,
// serving loops, harnesses that forbid hipMalloc). The two hopping terms read the source and
// write the result in the caller's arrays; the intermediate D src is kept in one static device
// array per GPU, where kq_mdaggm takes it from the allocator. The array's device address is looked
// up once per device with hipGetSymbolAddress (at the library's device set-up, or on the first call
// on another device); the name `kq_scratch` itself is never passed to a kernel.
// The work is queued on the library stream and the call returns without waiting
// (kq_synchronize waits for it).
// Calls on one GPU share the array: two calls that overlap on one GPU (from two
// host threads or two streams) race. Nothing in it has to start at zero: every
// byte a call reads was written earlier in the same call.
#include <string>

#include "kq_context.h"
#include "kq_solve.h"
#include "kuqcd_hip.h"

namespace kq {

// 64 MiB. The lattices the call accepts are those of which two vectors and one partial sum per 256
// sites fit (FP64: up to 32^4), the limit that the header states; the intermediate takes half of it.
constexpr size_t kNoAllocScratchBytes = (size_t)64 << 20;
static_assert(KQ_NOALLOC_SCRATCH_BYTES == kNoAllocScratchBytes, "header and library disagree on the scratch size");

__device__ __align__(256) unsigned char kq_scratch[kNoAllocScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
void *g_scratch[kMaxDevices] = {};

size_t round_up(size_t n) { return (n + 255) / 256 * 256; }

}  // namespace

void *noalloc_scratch()
{
    int dev = 0;
    KQ_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices)
        throw std::runtime_error("no-allocation scratch: device index out of range");
    if (g_scratch[dev] == nullptr) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(kq_scratch));
        if (e != hipSuccess || p == nullptr)
            throw std::runtime_error(std::string("hipGetSymbolAddress(kq_scratch) failed: ") + hipGetErrorString(e));
        g_scratch[dev] = p;
    }
    return g_scratch[dev];
}

static size_t noalloc_mdaggm_bytes(uint32_t Vh, size_t real_bytes)
{
    const size_t vec = round_up(2 * real_bytes * 3 * (size_t)Vh);
    return 2 * vec + round_up(sizeof(double) * ((Vh + 255) / 256)) + 256;
}

}  // namespace kq

using namespace kq;

extern "C" KuQCDStatus kq_mdaggm_noalloc(const void *src, void *dst, int parity, double sigma)
{
    try {
        if (src == nullptr || dst == nullptr) {
            set_error("src or dst is nullptr");
            return KUQCD_ERR_NULL_POINTER;
        }
        if (parity != 0 && parity != 1) {
            set_error("parity must be 0 (even) or 1 (odd)");
            return KUQCD_ERR_INVALID_PARAM;
        }
        const int slot = active_slot();
        if (slot < 0) {
            set_error("no init gauge_smeared and gauge_naik");
            return KUQCD_ERR_UNKNOWN_TYPE;
        }
        Context &c = ctx();
        const Geom g = slot_geom(slot);
        const bool dbl = c.fat[slot].prec == KUQCD_DOUBLE;
        const size_t real = dbl ? sizeof(double) : sizeof(float);
        const size_t need = noalloc_mdaggm_bytes(g.Vh, real);
        if (need > kNoAllocScratchBytes) {
            set_error("kq_mdaggm_noalloc: the loaded lattice needs " + std::to_string(need) +
                      " bytes of scratch, above the fixed " + std::to_string(kNoAllocScratchBytes) +
                      " (64 MiB: up to 32^4 sites in double precision); use kq_mdaggm");
            return KUQCD_ERR_INVALID_PARAM;
        }
        const size_t bytes = real * 6 * (size_t)g.Vh;
        // another GPU's memory too: its owner has made it accessible to this one
        if (!on_a_device(src) || !on_a_device(dst)) {
            set_error("kq_mdaggm_noalloc: src and dst must be device memory (kq_device_alloc / hipMalloc)");
            return KUQCD_ERR_INVALID_PARAM;
        }
        const char *a = static_cast<const char *>(src), *b = static_cast<const char *>(dst);
        if (a < b + bytes && b < a + bytes) {
            set_error("kq_mdaggm_noalloc: src and dst overlap");
            return KUQCD_ERR_INVALID_PARAM;
        }
        // the same link formats as kq_mdaggm (with_fp64_links), so the two agree bitwise
        if (dbl)
            with_fp64_links(slot, [&](auto fat, auto lng) {
                mdaggm_host<decltype(fat), decltype(lng), double>(
                    fat, lng, g, static_cast<const double *>(src), static_cast<double *>(dst),
                    static_cast<double2 *>(noalloc_scratch()), parity, sigma, c.stream);
            });
        else
            with_fp32_links(slot, [&](auto fat, auto lng) {
                mdaggm_host<decltype(fat), decltype(lng), float>(
                    fat, lng, g, static_cast<const float *>(src), static_cast<float *>(dst),
                    static_cast<float2 *>(noalloc_scratch()), parity, sigma, c.stream);
            });
        return KUQCD_SUCCESS;
    } catch (const std::exception &e) {
        set_error(e.what());
        return KUQCD_ERR_UNKNOWN_ERROR;
    }
}
