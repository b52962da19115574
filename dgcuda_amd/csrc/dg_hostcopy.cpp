// The runtime's copy of a pageable array goes through its own staging, one
// chunk at a time on one thread, and the first touch of a fresh destination
// (one fault per page) is taken on that thread too.  Here up to
// COPY_MAX_THREADS threads each take a contiguous part of the array through
// two pinned blocks of their own: while one block is on the bus the other is
// copied to or from the caller's memory.  Device to a fresh host array, 1 /
// 4 / 8 threads: 252 MB 19.4 / 8.3 / 7.4 ms, 42 MB 3.1 / 1.9 / 1.5, 6.3 MB
// 0.46 / 0.51 / 0.54: below COPY_MIN_PART bytes a part a second thread gains
// nothing, and four threads take most of the gain on a shared host.
#include "dg_hostcopy.h"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace dgmi {

namespace {

constexpr size_t COPY_BLOCK = PINNED_BLOCK_BYTES;
constexpr size_t COPY_MIN_PART = size_t(4) << 20;
constexpr int COPY_MAX_THREADS = 4;
constexpr size_t COPY_SMALL = size_t(64) << 10;
constexpr size_t COPY_IDLE_BLOCKS = 16;  // kept between calls, of all threads together (a server's set-up threads audit at a time)

// pinned blocks, shared by every thread of the process; at most
// COPY_IDLE_BLOCKS stay between calls, the others are freed
struct Blocks {
    std::mutex mu;
    std::vector<void*> idle;
    Blocks() { idle.reserve(COPY_IDLE_BLOCKS); }  // push_back never allocates
};
Blocks& blocks() {
    static Blocks* b = new Blocks();  // never destroyed: the runtime may be gone by then
    return *b;
}

hipError_t take_block(void** p) {
    {
        Blocks& b = blocks();
        std::lock_guard<std::mutex> lk(b.mu);
        if (!b.idle.empty()) {
            *p = b.idle.back();
            b.idle.pop_back();
            return hipSuccess;
        }
    }
    return hipHostMalloc(p, COPY_BLOCK, hipHostMallocPortable);
}

void give_block(void* p) {
    if (!p) return;
    {
        Blocks& b = blocks();
        std::lock_guard<std::mutex> lk(b.mu);
        if (b.idle.size() < COPY_IDLE_BLOCKS) {
            b.idle.push_back(p);
            return;
        }
    }
    (void)hipHostFree(p);
}

// One thread's part.  The blocks are idle again when it returns: on an error
// too, it waits for what it queued.
hipError_t copy_part(char* host, char* dev, size_t bytes, bool to_host, hipStream_t st) {
    void* blk[2] = {nullptr, nullptr};
    hipEvent_t ev[2] = {nullptr, nullptr};
    const size_t n = (bytes + COPY_BLOCK - 1) / COPY_BLOCK;
    constexpr int nb = 2;
    hipError_t e = hipSuccess;
    if (n == 1) {  // nothing to overlap: no events
        if ((e = take_block(&blk[0])) != hipSuccess) return e;
        if (!to_host) std::memcpy(blk[0], host, bytes);
        e = to_host ? hipMemcpyAsync(blk[0], dev, bytes, hipMemcpyDeviceToHost, st)
                    : hipMemcpyAsync(dev, blk[0], bytes, hipMemcpyHostToDevice, st);
        const hipError_t es = hipStreamSynchronize(st);
        if (e == hipSuccess) e = es;
        if (to_host && e == hipSuccess) std::memcpy(host, blk[0], bytes);
        give_block(blk[0]);
        return e;
    }
    for (int i = 0; i < nb && e == hipSuccess; i++) {
        e = take_block(&blk[i]);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming);
    }
    const auto len = [&](size_t i) { return std::min(COPY_BLOCK, bytes - i * COPY_BLOCK); };
    const auto queue = [&](size_t i) {
        const int b = (int)(i % nb);
        hipError_t q = to_host ? hipMemcpyAsync(blk[b], dev + i * COPY_BLOCK, len(i), hipMemcpyDeviceToHost, st)
                               : hipMemcpyAsync(dev + i * COPY_BLOCK, blk[b], len(i), hipMemcpyHostToDevice, st);
        return q == hipSuccess ? hipEventRecord(ev[b], st) : q;
    };
    if (to_host) {
        for (size_t i = 0; i < (size_t)nb && e == hipSuccess; i++) e = queue(i);
        for (size_t i = 0; i < n && e == hipSuccess; i++) {
            const int b = (int)(i % nb);
            e = hipEventSynchronize(ev[b]);
            if (e != hipSuccess) break;
            std::memcpy(host + i * COPY_BLOCK, blk[b], len(i));
            if (i + nb < n) e = queue(i + nb);
        }
    } else {
        for (size_t i = 0; i < n && e == hipSuccess; i++) {
            const int b = (int)(i % nb);
            if (i >= (size_t)nb) e = hipEventSynchronize(ev[b]);
            if (e != hipSuccess) break;
            std::memcpy(blk[b], host + i * COPY_BLOCK, len(i));
            e = queue(i);
        }
    }
    const hipError_t es = hipStreamSynchronize(st);
    if (e == hipSuccess) e = es;
    for (int i = 0; i < 2; i++) {
        if (ev[i]) (void)hipEventDestroy(ev[i]);
        give_block(blk[i]);
    }
    return e;
}

Status copy_parts(char* host, char* dev, size_t bytes, bool to_host, hipStream_t st) {
    if (bytes == 0) return hip_status(hipStreamSynchronize(st), "copy");
    const int parts = (int)std::min<size_t>(COPY_MAX_THREADS, std::max<size_t>(1, bytes / COPY_MIN_PART));
    if (parts == 1) return hip_status(copy_part(host, dev, bytes, to_host, st), "copy");
    // the parts run on streams of their own, so what `st` still has to do
    // to the device side is waited for here
    hipError_t e = hipStreamSynchronize(st);
    if (e != hipSuccess) return hip_status(e, "copy");
    int device = 0;
    if ((e = hipGetDevice(&device)) != hipSuccess) return hip_status(e, "copy");
    const size_t per = (bytes / parts + 63) / 64 * 64;
    std::vector<hipError_t> err(parts, hipSuccess);
    std::vector<hipStream_t> on(parts, nullptr);
    on[0] = st;
    for (int i = 1; i < parts; i++)
        if (!pool_stream(&on[i])) on[i] = nullptr;
    const auto part = [&](int i, hipStream_t s) {
        const size_t at = std::min(bytes, i * per), end = i + 1 == parts ? bytes : std::min(bytes, (i + 1) * per);
        if (at < end) err[i] = copy_part(host + at, dev + at, end - at, to_host, s);
    };
    std::vector<std::thread> th;
    std::vector<int> inline_parts;
    th.reserve(parts);  // (nothing may throw while a thread runs)
    inline_parts.reserve(parts);
    inline_parts.push_back(0);
    for (int i = 1; i < parts; i++) {
        bool started = false;
        if (on[i]) {
            try {
                th.emplace_back([&, i] {
                    err[i] = hipSetDevice(device);
                    if (err[i] == hipSuccess) part(i, on[i]);
                });
                started = true;
            } catch (const std::exception&) {  // no thread to be had: this one takes the part
            }
        }
        if (!started) inline_parts.push_back(i);
    }
    for (int i : inline_parts) part(i, st);
    for (std::thread& t : th) t.join();
    for (int i = 1; i < parts; i++) pool_release_stream(on[i]);
    for (hipError_t x : err)
        if (x != hipSuccess) return hip_status(x, "copy");
    return Status::ok();
}

}  // namespace

Status PinnedBlock::take() { return hip_status(take_block(&p), "pinned block"); }
PinnedBlock::~PinnedBlock() { give_block(p); }

Status copy_to_host(void* dst, const void* src_dev, size_t bytes, hipStream_t st) {
    return copy_parts((char*)dst, (char*)const_cast<void*>(src_dev), bytes, true, st);
}

Status upload_small(void* dst_dev, const void* src, size_t bytes, hipStream_t st) {
    if (bytes > COPY_SMALL) return copy_to_device(dst_dev, src, bytes, st);
    return hip_status(hipMemcpyAsync(dst_dev, src, bytes, hipMemcpyHostToDevice, st), "copy");
}

Status copy_to_device(void* dst_dev, const void* src, size_t bytes, hipStream_t st) {
    return copy_parts((char*)const_cast<void*>(src), (char*)dst_dev, bytes, false, st);
}

}  // namespace dgmi
