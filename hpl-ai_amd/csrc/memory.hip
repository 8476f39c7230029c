// memory.hip — device memory that outlives a call.
//
// Two kinds, both bounded and given back:
//  * StreamScratch (one per context): temporaries of the asynchronous entry
//    points, one buffer per stream.  An event marks the end of each use; the
//    next call waits for it on its own stream, which costs nothing where the
//    stream is the same (a destroyed stream's handle may come back as another
//    stream, so the handle alone proves no order).  No call waits on the host,
//    also where its buffer has to grow; a call that finds no room allocates in
//    stream order.  A stream-ordered
//    allocation per call instead stalls: on this runtime hipFreeAsync of
//    memory that an earlier call had freed waits for the device, which made
//    every second such call synchronous (18 us a call at least, 4 us as here).
//  * the block cache (one per device): the buffers of hplai_solve and
//    hplai_factor_f32, which are idle when those return.  Freeing tens of GB
//    costs the time to wipe them: hipFree of 40 GB takes 1.2 s once the
//    device's untouched memory is used up, more than the solve that used it.
#include <mutex>

#include "internal.hpp"

namespace hplai {

namespace {

constexpr int kMaxDevices = 64, kMaxIdle = 128;

struct Block {
    void *p;
    size_t bytes;
};

struct BlockCache {
    std::mutex mu;
    Block idle[kMaxIdle];   // oldest first
    int count = 0;
    size_t total = 0, bound = 0;
    int contexts = 0;
};

BlockCache g_cache[kMaxDevices];

// the caller holds c.mu
void trim_locked(BlockCache &c, size_t keep)
{
    int drop = 0;
    for (; c.total > keep && drop < c.count; ++drop) {
        (void)hipFree(c.idle[drop].p);
        c.total -= c.idle[drop].bytes;
    }
    for (int k = drop; k < c.count; ++k) c.idle[k - drop] = c.idle[k];
    c.count -= drop;
}

}  // namespace

// A context opens its device's cache; the last one to close it empties it.
// At most a sixth of the device's memory is kept.
int block_cache_open(int device, size_t device_bytes)
{
    HPLAI_CHECK(device >= 0 && device < kMaxDevices, "device %d out of range", device);
    BlockCache &c = g_cache[device];
    std::lock_guard<std::mutex> lock(c.mu);
    c.bound = device_bytes / 6;
    ++c.contexts;
    return HPLAI_OK;
}

void block_cache_close(int device)
{
    BlockCache &c = g_cache[device];
    std::lock_guard<std::mutex> lock(c.mu);
    if (--c.contexts == 0) trim_locked(c, 0);
}

// Every idle block back to the device; false if there was none.
bool block_cache_empty(int device)
{
    BlockCache &c = g_cache[device];
    std::lock_guard<std::mutex> lock(c.mu);
    const bool some = c.count > 0;
    trim_locked(c, 0);
    return some;
}

namespace {
// an allocation that empties the device's cache before it gives up
template <typename F>
hipError_t or_empty_cache(int device, F &&alloc)
{
    hipError_t e = alloc();
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        if (block_cache_empty(device)) e = alloc();
    }
    return e;
}
}  // namespace

hipError_t device_malloc(int device, void **p, size_t bytes)
{
    return or_empty_cache(device, [&] { return hipMalloc(p, bytes); });
}

// The smallest idle block of the size asked for or up to an eighth more, else
// new memory.  *bytes becomes the block's size, for block_free.
hipError_t block_alloc(int device, void **p, size_t *bytes)
{
    BlockCache &c = g_cache[device];
    {
        std::lock_guard<std::mutex> lock(c.mu);
        int best = -1;
        for (int k = 0; k < c.count; ++k)
            if (c.idle[k].bytes >= *bytes && c.idle[k].bytes <= *bytes + *bytes / 8 &&
                (best < 0 || c.idle[k].bytes < c.idle[best].bytes))
                best = k;
        if (best >= 0) {
            *p = c.idle[best].p;
            *bytes = c.idle[best].bytes;
            c.total -= *bytes;
            for (int k = best + 1; k < c.count; ++k) c.idle[k - 1] = c.idle[k];
            --c.count;
            return hipSuccess;
        }
    }
    return device_malloc(device, p, *bytes);
}

namespace {
// into the cache if it has room for the block; the caller holds c.mu
bool put_locked(BlockCache &c, void *p, size_t bytes)
{
    if (c.contexts == 0 || c.count == kMaxIdle || c.total + bytes > c.bound) return false;
    c.idle[c.count++] = Block{p, bytes};
    c.total += bytes;
    return true;
}
}  // namespace

// p must be idle on the device.  Older blocks make room; freeing one waits for the device.
void block_free(int device, void *p, size_t bytes)
{
    if (p == nullptr) return;
    BlockCache &c = g_cache[device];
    {
        std::lock_guard<std::mutex> lock(c.mu);
        if (c.contexts > 0 && bytes <= c.bound) trim_locked(c, c.bound - bytes);
        if (put_locked(c, p, bytes)) return;
    }
    (void)hipFree(p);
}

// The same without a wait: false, and p still the caller's, if there is no room.
bool block_put(int device, void *p, size_t bytes)
{
    BlockCache &c = g_cache[device];
    std::lock_guard<std::mutex> lock(c.mu);
    return put_locked(c, p, bytes);
}

// ---------------------------------------------------------------------------

ScratchLease::ScratchLease(hplai_ctx ctx, hipStream_t stream, size_t bytes) : stream_(stream)
{
    if (bytes == 0) return;
    StreamScratch &sc = ctx->pool;
    // a captured call needs memory of its own: its graph may run beside later
    // calls on this stream
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    const bool eager = hipStreamIsCapturing(stream, &cap) == hipSuccess && cap == hipStreamCaptureStatusNone;
    if (eager && bytes <= kScratchMax) {
        // held until the call's kernels are enqueued: no other call on this
        // context can put its own between them
        lock_ = std::unique_lock<std::mutex>(sc.mu);
        StreamScratch::Entry *e = sc.find(stream);
        hipError_t err = hipSuccess;
        if (e != nullptr && e->bytes >= bytes)
            err = hipStreamWaitEvent(stream, e->done, 0);
        else
            e = sc.replace(ctx->device, e, stream, bytes, &err);
        if (err != hipSuccess) {
            rc = hip_fail(err, "scratch memory");
            return;
        }
        if (e != nullptr) {
            ptr = e->p;
            done_ = e->done;
            return;
        }
        lock_.unlock();   // no room: this call's own
    }
    (void)hipGetLastError();
    auto alloc = [&] { return hipMallocAsync(&ptr, bytes, stream); };
    const hipError_t err = eager ? or_empty_cache(ctx->device, alloc) : alloc();
    if (err != hipSuccess) {
        ptr = nullptr;
        rc = hip_fail(err, "hipMallocAsync scratch");
        return;
    }
    async_ = true;
}

ScratchLease::~ScratchLease()
{
    if (async_) (void)hipFreeAsync(ptr, stream_);
    if (done_ != nullptr) (void)hipEventRecord(done_, stream_);
}

StreamScratch::Entry *StreamScratch::find(hipStream_t stream)
{
    for (int k = 0; k < count; ++k)
        if (entries[k].owned && entries[k].stream == stream) return &entries[k];
    return nullptr;
}

// A buffer of at least `bytes` for `stream` in place of `old` (may be NULL),
// which is outgrown: its memory may be in use until its event has passed.  No
// work is waited for: buffers that are done with go back to the block cache
// where it has room, or to the call if they fit; NULL without an error if all
// others are in use.
StreamScratch::Entry *StreamScratch::replace(int device, Entry *old, hipStream_t stream, size_t bytes, hipError_t *err)
{
    // allocating and asking for events is legal beside another stream's capture only so
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    Entry *fit = nullptr;
    if (old != nullptr) old->owned = false;
    size_t want = size_t(1) << 20;
    while (want < bytes) want *= 2;
    // twice: buffers without a stream, then, if there is no room yet, other streams' as well
    for (int pass = 0; pass < 2 && fit == nullptr; ++pass) {
        if (pass == 1 && total + want <= kTotal && count < kMax) break;
        for (int k = count - 1; k >= 0 && fit == nullptr; --k) {
            Entry &e = entries[k];
            if ((pass == 0 && e.owned) || hipEventQuery(e.done) != hipSuccess) continue;
            if (e.bytes >= want) {
                fit = &e;
            } else if (block_put(device, e.p, e.bytes)) {
                (void)hipEventDestroy(e.done);
                total -= e.bytes;
                e = entries[--count];
            }
        }
    }
    (void)hipGetLastError();   // hipErrorNotReady
    if (fit == nullptr && total + want <= kTotal && count < kMax) {
        Entry n{stream, nullptr, nullptr, want, true};
        *err = hipEventCreateWithFlags(&n.done, hipEventDisableTiming);
        if (*err == hipSuccess) *err = block_alloc(device, &n.p, &n.bytes);
        if (*err == hipSuccess) {
            fit = &entries[count++];
            *fit = n;
            total += n.bytes;
        } else if (n.done != nullptr) {
            (void)hipEventDestroy(n.done);
        }
    }
    if (fit != nullptr) {
        fit->stream = stream;
        fit->owned = true;
    }
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    return fit;
}

// Everything back, after the work enqueued on it.
void StreamScratch::clear(int device)
{
    for (; count > 0; --count) {
        Entry &e = entries[count - 1];
        (void)hipEventSynchronize(e.done);
        (void)hipEventDestroy(e.done);
        block_free(device, e.p, e.bytes);
    }
    total = 0;
}

}  // namespace hplai
