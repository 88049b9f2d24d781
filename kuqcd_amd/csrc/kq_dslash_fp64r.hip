// Hopping-term instantiations: FP64 fat links with FP64 long links in 14 reals.
#include "kq_dslash_impl.h"

namespace kq {

template uint32_t launch_dslash<LinkD, LinkD14, double>(DslashArgs<LinkD, LinkD14, double>, int, int, int, hipStream_t,
                                                    int);
template void launch_dslash_host<LinkD, LinkD14, double>(const DslashArgs<LinkD, LinkD14, double> &, int, int, int, hipStream_t);
template void launch_dslash_p<LinkD, LinkD14, double>(DslashArgs<LinkD, LinkD14, double>, CgmState<double> *, const c2_t<double> *, Vec<double>, Vec<double>,
                                              const double *, uint32_t, double *, hipStream_t);

}  // namespace kq
