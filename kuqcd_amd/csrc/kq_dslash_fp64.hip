// Hopping-term instantiations: FP64 links.
#include "kq_dslash_impl.h"

namespace kq {

template uint32_t launch_dslash<LinkD, LinkD, double>(DslashArgs<LinkD, LinkD, double>, int, int, int, hipStream_t, int);
template void launch_dslash_host<LinkD, LinkD, double>(const DslashArgs<LinkD, LinkD, double> &, int, int, int, hipStream_t);
template void launch_dslash_p<LinkD, LinkD, double>(DslashArgs<LinkD, LinkD, double>, CgmState<double> *, const c2_t<double> *, Vec<double>, Vec<double>,
                                              const double *, uint32_t, double *, hipStream_t);

}  // namespace kq
