// P on FP32 vectors: the Krylov steps.
#include "stencil_impl.hpp"

namespace mfd {
#define MFD_APPLY(R, MODE, EPI)                                                                                      \
    template int launch_apply<R, MODE, EPI>(mfd_op *, const cx<R> *, cx<R> *, const c64 *, int64_t, double *, Scal *, \
                                            double *, const int *, hipEvent_t, bool)
MFD_APPLY(float, MODE_P, EPI_DOT);
template void launch_cocg_stencil<float>(mfd_op *, dim3, int, int, int, int, const cx<float> *, cx<float> *, const cx<float> *, cx<float> *,
                                       cx<float> *);
}  // namespace mfd
