// Hopping-term instantiations: FP32 links (18-real long links and 12-real LinkF12).
#include "kq_dslash_impl.h"

namespace kq {

template uint32_t launch_dslash<LinkF, LinkF, float>(DslashArgs<LinkF, LinkF, float>, int, int, int, hipStream_t, int);
template uint32_t launch_dslash<LinkF, LinkF12, float>(DslashArgs<LinkF, LinkF12, float>, int, int, int, hipStream_t, int);
template void launch_dslash_host<LinkF, LinkF, float>(const DslashArgs<LinkF, LinkF, float> &, int, int, int, hipStream_t);
template void launch_dslash_host<LinkF, LinkF12, float>(const DslashArgs<LinkF, LinkF12, float> &, int, int, int, hipStream_t);
template void launch_dslash_p<LinkF, LinkF, float>(DslashArgs<LinkF, LinkF, float>, CgmState<float> *, const c2_t<float> *, Vec<float>, Vec<float>,
                                              const double *, uint32_t, double *, hipStream_t);
template void launch_dslash_p<LinkF, LinkF12, float>(DslashArgs<LinkF, LinkF12, float>, CgmState<float> *, const c2_t<float> *, Vec<float>, Vec<float>,
                                              const double *, uint32_t, double *, hipStream_t);

}  // namespace kq
