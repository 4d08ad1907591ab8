// SQMR steps of a problem that fits the chip, in one resident kernel.
#pragma once
#include "krylov_dev.hpp"

namespace mfd {

// Whether nrhs right-hand sides of the operator's system run resident with
// vectors of storage precision R: the stencil form is built (diagonal or full
// ε with μ = 1, or μ ≠ 1 with diagonal ε; any boundft, a component window),
// every box of one right-hand side has a place on the chip at once, and the
// launches that nrhs of them take are faster than the step-by-step kernels
// (chunk: steps between two looks at the scalars).
template <typename R>
bool resident_ok(const mfd_op *op, int64_t nrhs, int chunk);

// the boxes it runs in, to stderr
template <typename R>
void resident_trace(const mfd_op *op);

// Runs up to `steps` SQMR steps on the operator's workspace, on its stream;
// the state before and after is that between steps (r, q, d, z and the
// scalars).  After each `chunk` steps a right-hand side also stops when its
// τ ≤ near·‖c‖.
template <typename R>
int resident_steps(mfd_op *op, int64_t nrhs, int steps, int chunk, double near);

// Scal::stag of a right-hand side whose blocks gave up waiting for each other;
// what resident_steps returns when the launch was refused (fewer places than the
// device reported, or another process holds its cooperative queue): the state is
// still that between steps, resident_ok is false for the context's operators for
// some seconds, and the step-by-step kernels go on
enum { RESIDENT_TIMEOUT = -1, RESIDENT_REFUSED = -2 };

}  // namespace mfd
