// Scratch device memory of a context, and copies between host and device.
#include "ctxmem.hpp"
#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

namespace mfd {

// An allocation and its release cost 60–800 µs of a call (the release waits
// for the device and unmaps the pages), so blocks are kept from call to call:
// 0.1% of the device's memory at most.  A call whose arrays need more (an
// assembly of more than some 200,000 cells) allocates as it did, beside tens of
// ms of copies (90×80×70: 29 ms).
constexpr size_t CTXMEM_KEEP = 256u << 20;
constexpr int NBLK = 32;

// Large copies to and from pageable memory run at 7–12 GB/s: one host thread
// moves the data between the caller's pages and the runtime's staging memory.
// Here a thread per 4 MB does that (eight at most), each with two pinned slots
// of its own, so that one slot fills while the other drains.  The assembled
// 56×48×50 A (126 MB out) takes 17.1 ms the plain way and 10.5, 9.8 and 8.7 ms
// with 2, 4 and 8 threads.  Below 16 MB (four threads' worth) the plain way stays:
// an apply with 11 MB in and out would gain 0.2 of 1.3 ms, but the pages that the
// threads touch first end up on other NUMA nodes, and a caller that goes through
// them afterwards loses more (a 2D solve that reorders 11 MB: 1 of 11 ms).
constexpr int COPY_THREADS = 8;
constexpr size_t CHUNK = 1u << 20;
constexpr size_t PER_THREAD = 4u << 20;
constexpr size_t COPY_MIN = 4 * PER_THREAD;

struct CtxMem {
    int device;
    std::mutex m;         // the blocks
    struct {
        void *p = nullptr;
        size_t bytes = 0;
        bool used = false;
    } blk[NBLK];
    hipStream_t side = nullptr;   // (under m)
    std::mutex copying;   // the slots
    char *pin = nullptr;
    hipEvent_t ev[2 * COPY_THREADS] = {};
};

CtxMem *ctxmem_create(int device) {
    CtxMem *m = new (std::nothrow) CtxMem();
    if (m) m->device = device;
    return m;
}

static void drop_unused(CtxMem *m) {
    for (auto &b : m->blk)
        if (b.p && !b.used) {
            hipFree(b.p);
            b.p = nullptr;
            b.bytes = 0;
        }
}

void ctxmem_destroy(CtxMem *m) {
    if (!m) return;
    drop_unused(m);
    if (m->side) hipStreamDestroy(m->side);
    for (auto &e : m->ev)
        if (e) hipEventDestroy(e);
    if (m->pin) hipHostFree(m->pin);
    delete m;
}

hipError_t ctx_malloc(mfd_ctx *ctx, void **p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipErrorOutOfMemory) return e;
    {
        std::lock_guard<std::mutex> lock(ctx->mem->m);
        drop_unused(ctx->mem);
    }
    hipGetLastError();   // the failure is not reported if the second try succeeds
    return hipMalloc(p, bytes);
}

int scratch_get(mfd_ctx *ctx, size_t bytes, void **p) {
    if (bytes > SIZE_MAX - 65535) {   // (a wrapped size is not a small one)
        *p = nullptr;
        set_error("scratch size out of range");
        return MFD_ERR_ALLOC;
    }
    bytes = (std::max<size_t>(bytes, 1) + 65535) / 65536 * 65536;
    CtxMem *m = ctx->mem;
    {
        std::lock_guard<std::mutex> lock(m->m);
        int best = -1;
        for (int i = 0; i < NBLK; ++i) {
            const auto &b = m->blk[i];
            if (b.p && !b.used && b.bytes >= bytes && b.bytes <= 2 * bytes && (best < 0 || b.bytes < m->blk[best].bytes)) best = i;
        }
        if (best >= 0) {
            m->blk[best].used = true;
            *p = m->blk[best].p;
            return MFD_OK;
        }
    }
    *p = nullptr;
    if (ctx_malloc(ctx, p, bytes) != hipSuccess) {
        *p = nullptr;
        set_error("hipMalloc failed");
        return MFD_ERR_ALLOC;
    }
    std::lock_guard<std::mutex> lock(m->m);
    for (auto &b : m->blk)
        if (!b.p) {
            b.p = *p;
            b.bytes = bytes;
            b.used = true;
            break;
        }
    return MFD_OK;   // no room in the table: released when put back
}

void scratch_put(mfd_ctx *ctx, void *p) {
    CtxMem *m = ctx->mem;
    void *drop[NBLK + 1];
    int nd = 0;
    {
        std::lock_guard<std::mutex> lock(m->m);
        int at = -1;
        size_t unused = 0;
        for (int i = 0; i < NBLK; ++i) {
            auto &b = m->blk[i];
            if (b.p == p) {
                b.used = false;
                at = i;
            }
            if (b.p && !b.used) unused += b.bytes;
        }
        if (at < 0) drop[nd++] = p;
        // over the bound: the others go first, then this one
        for (int k = 0; k <= NBLK && unused > CTXMEM_KEEP; ++k) {
            const int i = k < NBLK ? k : at;
            if (i < 0 || (k < NBLK && i == at)) continue;
            auto &b = m->blk[i];
            if (!b.p || b.used) continue;
            unused -= b.bytes;
            drop[nd++] = b.p;
            b.p = nullptr;
            b.bytes = 0;
        }
    }
    for (int i = 0; i < nd; ++i) hipFree(drop[i]);   // waits for the device
}

hipStream_t ctx_side_stream(mfd_ctx *ctx) {
    CtxMem *m = ctx->mem;
    std::lock_guard<std::mutex> lock(m->m);
    if (!m->side && hipStreamCreateWithFlags(&m->side, hipStreamNonBlocking) != hipSuccess) {
        hipGetLastError();
        m->side = nullptr;
    }
    return m->side;
}

static bool slots_ready(CtxMem *m) {
    if (m->pin) return true;
    for (auto &e : m->ev)
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            e = nullptr;
            hipGetLastError();
            return false;
        }
    if (hipHostMalloc((void **)&m->pin, 2 * COPY_THREADS * CHUNK, hipHostMallocDefault) != hipSuccess) {
        m->pin = nullptr;
        hipGetLastError();
        return false;
    }
    return true;
}

// chunks w, w + nt, … of the copy, through thread w's two slots
static hipError_t copy_chunks(CtxMem *m, hipStream_t s, char *dst, const char *src, size_t bytes, bool in, int w, int nt) {
    const int64_t nc = (int64_t)((bytes + CHUNK - 1) / CHUNK);
    auto size = [&](int64_t c) { return std::min(CHUNK, bytes - (size_t)c * CHUNK); };
    auto slot = [&](int64_t c) { return 2 * w + (int)((c / nt) & 1); };
    hipError_t e = hipSuccess;
    if (in) {
        for (int64_t c = w; c < nc && e == hipSuccess; c += nt) {
            const int k = slot(c);
            char *pin = m->pin + (size_t)k * CHUNK;
            e = hipEventSynchronize(m->ev[k]);   // the slot's last copy, this call's or an earlier one's
            if (e != hipSuccess) break;
            memcpy(pin, src + (size_t)c * CHUNK, size(c));
            e = hipMemcpyAsync(dst + (size_t)c * CHUNK, pin, size(c), hipMemcpyHostToDevice, s);
            if (e == hipSuccess) e = hipEventRecord(m->ev[k], s);
        }
        return e;
    }
    auto issue = [&](int64_t c) {
        const int k = slot(c);
        hipError_t r = hipMemcpyAsync(m->pin + (size_t)k * CHUNK, src + (size_t)c * CHUNK, size(c), hipMemcpyDeviceToHost, s);
        return r == hipSuccess ? hipEventRecord(m->ev[k], s) : r;
    };
    if (w < nc) e = issue(w);
    for (int64_t c = w; c < nc && e == hipSuccess; c += nt) {
        if (c + nt < nc) e = issue(c + nt);
        const hipError_t r = hipEventSynchronize(m->ev[slot(c)]);
        if (r != hipSuccess) return r;
        memcpy(dst + (size_t)c * CHUNK, m->pin + (size_t)slot(c) * CHUNK, size(c));
    }
    return e;
}

static int copy(mfd_ctx *ctx, void *dst, const void *src, size_t bytes, bool in) {
    CtxMem *m = ctx->mem;
    hipStream_t s = ctx->stream;
    hipError_t e = hipSuccess;
    std::unique_lock<std::mutex> lock(m->copying, std::defer_lock);
    // another thread's copy on this context is using the slots: the plain way
    if (bytes < COPY_MIN || !lock.try_lock() || !slots_ready(m)) {
        e = hipMemcpyAsync(dst, src, bytes, in ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, s);
        if (!in && e == hipSuccess) e = hipStreamSynchronize(s);
    } else {
        const int nt = (int)std::min<size_t>(COPY_THREADS, bytes / PER_THREAD);
        std::atomic<int> err{(int)hipSuccess};
        auto part = [&](int w) {
            hipError_t r = hipSetDevice(m->device);
            if (r == hipSuccess) r = copy_chunks(m, s, (char *)dst, (const char *)src, bytes, in, w, nt);
            if (r != hipSuccess) err = (int)r;
        };
        std::thread th[COPY_THREADS];
        int started = 1;
        try {
            for (; started < nt; ++started) th[started] = std::thread(part, started);
        } catch (...) {   // no more threads: the rest here
        }
        part(0);
        for (int w = started; w < nt; ++w) part(w);
        for (int w = 1; w < started; ++w) th[w].join();
        e = (hipError_t)err.load();
        if (!in) {
            const hipError_t r = hipStreamSynchronize(s);
            if (e == hipSuccess) e = r;
        } else if (e != hipSuccess) {
            hipStreamSynchronize(s);   // nothing of a failed copy stays queued on the slots
        }
    }
    if (e != hipSuccess) {
        set_error(std::string(in ? "copy to device failed: " : "copy to host failed: ") + hipGetErrorString(e));
        return MFD_ERR_HIP;
    }
    return MFD_OK;
}

int copy_in(mfd_ctx *ctx, void *dst, const void *src, size_t bytes) { return bytes ? copy(ctx, dst, src, bytes, true) : MFD_OK; }
int copy_out(mfd_ctx *ctx, void *dst, const void *src, size_t bytes) {
    if (bytes) return copy(ctx, dst, src, bytes, false);
    return hipStreamSynchronize(ctx->stream) == hipSuccess ? MFD_OK : MFD_ERR_HIP;
}

}  // namespace mfd
