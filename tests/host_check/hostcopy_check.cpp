// The copies between host arrays and device memory, from several caller
// threads at a time against the model of the runtime: every byte arrives, on
// either side of a block and of one to four parts; with each runtime call
// failing in turn the copy returns an error or the right bytes, and leaves no
// event, no stream and no more than the pool's blocks behind.
#include <cstdio>

#include "model_pool.h"
#include "dg_hostcopy.h"

#ifdef NO_THREADS  // threads are refused while set (a build without sanitizers, which have their own)
#include <dlfcn.h>
#include <errno.h>
static std::atomic<bool> refuse{false};
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) noexcept {
    static const auto real = (int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*))dlsym(RTLD_NEXT, "pthread_create");
    return refuse ? EAGAIN : real(t, a, f, x);
}
#endif

using namespace dgmi;

namespace {

constexpr size_t MB = size_t(1) << 20;
constexpr int IDLE_BLOCKS = 16;

std::vector<char> bytes_of(size_t n, unsigned seed) {
    std::vector<char> v(n);
    unsigned x = seed * 2654435761u + 1;
    for (char& c : v) c = (char)((x = x * 1664525u + 1013904223u) >> 24);
    return v;
}

// one copy in and one out; false if either returned an error
bool trip(size_t n, unsigned seed, bool check) {
    hipStream_t st = nullptr;
    if (!pool_stream(&st)) return false;
    const std::vector<char> a = bytes_of(n, seed);
    std::vector<char> dev(n, 0), b(n, 1);
    const Status in = copy_to_device(dev.data(), a.data(), n, st);
    const Status out = copy_to_host(b.data(), dev.data(), n, st);
    S(st)->wait();
    pool_release_stream(st);
    if (in && (check || out)) CHECK(dev == a);
    if (in && out) CHECK(b == a);
    return in && out;
}

}  // namespace

int main(int argc, char**) {
    const bool brief = argc > 1;  // under a thread sanitizer: fewer sizes
    std::vector<size_t> sizes = {0, 1, 8 * 63, MB - 8, MB, MB + 8, 2 * MB, 2 * MB + 8, 3 * MB + 1, 8 * MB - 8, 8 * MB,
                                 8 * MB + 8, 12 * MB - 8, 12 * MB, 12 * MB + 8, 16 * MB - 8, 16 * MB, 16 * MB + 72, 21 * MB + 5};
    if (brief) sizes = {8 * 63, MB, MB + 8, 8 * MB - 8, 8 * MB, 12 * MB + 8, 16 * MB + 72};
    for (size_t n : sizes) CHECK(trip(n, 1, true));
#ifdef NO_THREADS
    refuse = true;  // (the pool's streams are there)
    for (size_t n : sizes) CHECK(trip(n, 1, true));
    refuse = false;
#endif
    std::vector<std::thread> th;
    for (unsigned i = 0; i < 4; i++)
        th.emplace_back([&, i] {
            for (size_t k = 0; k < sizes.size(); k++) CHECK(trip(sizes[(k + 3 * i) % sizes.size()], i + 2, true));
        });
    for (std::thread& t : th) t.join();
    th.clear();
    for (unsigned i = 0; i < 24; i++)  // more blocks out at a time than stay idle
        th.emplace_back([&, i] {
            for (int k = 0; k < 20; k++) {
                PinnedBlock b;
                CHECK(b.take());
                for (int j = 0; j < 64; j++) b.data()[j] = i;
                std::this_thread::yield();
                for (int j = 0; j < 64; j++) CHECK(b.data()[j] == i);
            }
        });
    for (std::thread& t : th) t.join();
    CHECK(model::host_blocks <= IDLE_BLOCKS && model::events == 0);
    CHECK(stream_pool().idle() == stream_pool().all.size());
    if (!brief)
        for (size_t n : {8 * (size_t)63, 2 * MB + 8, 8 * MB + 8}) {
            int failed = 0;
            for (long at = 0;; at++) {
                model::calls = 0;
                model::fail_at = at;
                failed += !trip(n, 7, false);
                const bool reached = model::calls > at;
                model::fail_at = -1;
                CHECK(model::host_blocks <= IDLE_BLOCKS && model::events == 0);
                CHECK(stream_pool().idle() == stream_pool().all.size());
                CHECK(trip(n, 9, true));  // whole again
                if (!reached) break;
            }
            CHECK(failed > 0);
        }
    std::printf("host copies ok\n");
    return 0;
}
