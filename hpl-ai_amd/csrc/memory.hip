// memory.hip — device memory that outlives a call.
//
// Two kinds, both bounded and given back:
//  * StreamScratch (one per context): temporaries of the asynchronous entry
//    points, one buffer per stream.  An event marks the end of each use; the
//    next call waits for it on its own stream, which costs nothing where the
//    stream is the same (a destroyed stream's handle may come back as another
//    stream, so the handle alone proves no order).  A stream-ordered
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

// p must be idle on the device.
void block_free(int device, void *p, size_t bytes)
{
    if (p == nullptr) return;
    BlockCache &c = g_cache[device];
    {
        std::lock_guard<std::mutex> lock(c.mu);
        if (c.contexts > 0 && bytes <= c.bound) {
            trim_locked(c, c.bound - bytes);
            if (c.count < kMaxIdle) {
                c.idle[c.count++] = Block{p, bytes};
                c.total += bytes;
                return;
            }
        }
    }
    (void)hipFree(p);
}

// ---------------------------------------------------------------------------

namespace {
// per context: kept in all, and the largest buffer kept
constexpr size_t kScratchTotal = size_t(1) << 30;
}  // namespace

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
        StreamScratch::Entry *e = nullptr;
        for (int k = 0; k < sc.count; ++k)
            if (sc.entries[k].stream == stream) e = &sc.entries[k];
        if (e == nullptr || e->bytes < bytes) {
            size_t want = size_t(1) << 20;
            while (want < bytes) want *= 2;
            if (e != nullptr) sc.drop(ctx->device, e);   // outgrown
            // buffers of many streams, some of them gone
            if (sc.total + want > kScratchTotal || sc.count == StreamScratch::kMax) sc.clear(ctx->device);
            StreamScratch::Entry n{stream, nullptr, nullptr, want};
            hipError_t err = hipEventCreateWithFlags(&n.done, hipEventDisableTiming);
            if (err == hipSuccess) err = block_alloc(ctx->device, &n.p, &n.bytes);
            if (err != hipSuccess) {
                if (n.done != nullptr) (void)hipEventDestroy(n.done);
                rc = hip_fail(err, "scratch memory");
                return;
            }
            e = &sc.entries[sc.count++];
            *e = n;
            sc.total += n.bytes;
        } else {
            const hipError_t err = hipStreamWaitEvent(stream, e->done, 0);
            if (err != hipSuccess) {
                rc = hip_fail(err, "hipStreamWaitEvent scratch");
                return;
            }
        }
        ptr = e->p;
        done_ = e->done;
        return;
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

void StreamScratch::drop(int device, Entry *e)
{
    (void)hipEventSynchronize(e->done);
    (void)hipEventDestroy(e->done);
    block_free(device, e->p, e->bytes);
    total -= e->bytes;
    *e = entries[--count];
}

void StreamScratch::clear(int device)
{
    while (count > 0) drop(device, &entries[count - 1]);
}

}  // namespace hplai
