// Scratch device memory of a context, and copies between host and device.
#pragma once
#include "common.hpp"

namespace mfd {

struct CtxMem;
CtxMem *ctxmem_create(int device);   // null: out of memory
void ctxmem_destroy(CtxMem *m);      // gives everything back

// Device memory for the length of a call, ordered by the context's stream (a
// block handed on may still be in use by work queued before).  Blocks come
// from those the context keeps: at most CTXMEM_KEEP bytes while unused, given
// back when an allocation fails and when the context ends.
int scratch_get(mfd_ctx *ctx, size_t bytes, void **p);
void scratch_put(mfd_ctx *ctx, void *p);
struct Scratch {
    mfd_ctx *ctx = nullptr;
    void *p = nullptr;
    int get(mfd_ctx *c, size_t bytes) {
        ctx = c;
        return scratch_get(c, bytes, &p);
    }
    ~Scratch() {
        if (p) scratch_put(ctx, p);
    }
    Scratch() = default;
    Scratch(const Scratch &) = delete;
    Scratch &operator=(const Scratch &) = delete;
};
// hipMalloc that gives the context's unused blocks back before it fails
hipError_t ctx_malloc(mfd_ctx *ctx, void **p, size_t bytes);

// The context's second stream, made when first asked for (null: it could not be).
// Work there is forked from and joined to the context's stream by events, so that
// nothing else needs to know of it.
hipStream_t ctx_side_stream(mfd_ctx *ctx);

// Copies on the context's stream.  src of copy_in stays the caller's until the
// stream is waited for; copy_out has written dst (and waited for the stream).
int copy_in(mfd_ctx *ctx, void *dst, const void *src, size_t bytes);
int copy_out(mfd_ctx *ctx, void *dst, const void *src, size_t bytes);

}  // namespace mfd
