// P on FP64 vectors: the Krylov steps.
#include "stencil_impl.hpp"

namespace mfd {
#define MFD_APPLY(R, MODE, EPI)                                                                                      \
    template int launch_apply<R, MODE, EPI>(mfd_op *, const cx<R> *, cx<R> *, const c64 *, int64_t, double *, Scal *, \
                                            double *, const int *, hipEvent_t, bool)
MFD_APPLY(double, MODE_P, EPI_DOT);
template void launch_finish<EPI_DOT>(hipStream_t, int, int64_t, double *, Scal *, double *, const int *);
template void launch_cocg_stencil<double>(mfd_op *, dim3, int, int, int, int, const cx<double> *, cx<double> *, const cx<double> *, cx<double> *,
                                       cx<double> *);
}  // namespace mfd
