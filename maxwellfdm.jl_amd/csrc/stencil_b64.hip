// P on FP64 vectors: the two products of a BiCGSTAB step.
#include "stencil_impl.hpp"

namespace mfd {
#define MFD_APPLY(R, MODE, EPI)                                                                                      \
    template int launch_apply<R, MODE, EPI>(mfd_op *, const cx<R> *, cx<R> *, const c64 *, int64_t, double *, Scal *, \
                                            double *, const int *, hipEvent_t, bool)
MFD_APPLY(double, MODE_P, EPI_BDOT);
MFD_APPLY(double, MODE_P, EPI_XDOT);
}  // namespace mfd
