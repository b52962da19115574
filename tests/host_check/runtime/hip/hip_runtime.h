// A model of the runtime's host side, for checks of the host code on the
// CPU: each stream is a thread that runs its queue in order, so copies and
// events are as asynchronous as the runtime's; memory is the host's.  What
// the runtime does not order is not ordered here either, so that a thread
// sanitizer sees it.  fail_at makes the call of that number fail.
#pragma once
#include "../../hip/hip_runtime.h"
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <deque>
#include <functional>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

enum { hipErrorOutOfMemory = 2, hipErrorInvalidValue = 1 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum { hipHostMallocPortable = 1, hipEventDisableTiming = 2, hipStreamCaptureModeThreadLocal = 1 };
inline const char* hipGetErrorString(hipError_t) { return "model error"; }

namespace model {

struct Stream {
    std::mutex mu;
    std::condition_variable cv;
    std::deque<std::function<void()>> q;
    bool busy = false, stop = false;
    std::atomic<bool> capturing{false};
    int captured = 0;  // steps put on it while it is captured
    int device = 0;
    std::thread th;
    Stream() : th([this] { loop(); }) {}
    ~Stream() {
        {
            std::lock_guard<std::mutex> lk(mu);
            stop = true;
        }
        cv.notify_all();
        th.join();
    }
    void loop() {
        std::unique_lock<std::mutex> lk(mu);
        while (true) {
            cv.wait(lk, [&] { return stop || !q.empty(); });
            if (q.empty()) return;
            auto f = std::move(q.front());
            q.pop_front();
            busy = true;
            lk.unlock();
            f();
            lk.lock();
            busy = false;
            cv.notify_all();
        }
    }
    void put(std::function<void()> f) {
        {
            std::lock_guard<std::mutex> lk(mu);
            q.push_back(std::move(f));
        }
        cv.notify_all();
    }
    void wait() {
        std::unique_lock<std::mutex> lk(mu);
        cv.wait(lk, [&] { return q.empty() && !busy; });
    }
};

struct Event {
    std::mutex mu;
    std::condition_variable cv;
    long recorded = 0, reached = 0;
};

inline std::atomic<long> calls{0}, fail_at{-1}, host_blocks{0}, events{0};
inline bool fails() { return calls.fetch_add(1) == fail_at.load(); }

}  // namespace model

typedef std::shared_ptr<model::Event>* hipEvent_t;
inline model::Stream* S(hipStream_t s) { return static_cast<model::Stream*>(s); }

typedef int hipDevice_t;
namespace model {
inline thread_local int device = 0;
}
inline hipError_t hipGetDevice(int* d) { *d = model::device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) {
    if (model::fails()) return hipErrorInvalidValue;
    model::device = d;
    return hipSuccess;
}
inline hipError_t hipStreamGetDevice(hipStream_t st, hipDevice_t* d) {
    if (model::fails()) return hipErrorInvalidValue;
    *d = S(st)->device;
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, int) {
    if (model::fails()) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    model::host_blocks++;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
    std::free(p);
    model::host_blocks--;
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    if (model::fails()) return hipErrorInvalidValue;
    S(st)->put([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
// (a wait that fails has waited all the same)
inline hipError_t hipStreamSynchronize(hipStream_t st) {
    const bool bad = model::fails() || S(st)->capturing.load();
    S(st)->wait();
    return bad ? hipErrorInvalidValue : hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) {
    if (model::fails()) return hipErrorOutOfMemory;
    *e = new std::shared_ptr<model::Event>(new model::Event());
    model::events++;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
    if (model::fails()) return hipErrorInvalidValue;
    std::shared_ptr<model::Event> ev = *e;
    long n;
    {
        std::lock_guard<std::mutex> lk(ev->mu);
        n = ++ev->recorded;
    }
    S(st)->put([ev, n] {
        std::lock_guard<std::mutex> lk(ev->mu);
        ev->reached = n;
        ev->cv.notify_all();
    });
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    std::shared_ptr<model::Event> ev = *e;
    std::unique_lock<std::mutex> lk(ev->mu);
    ev->cv.wait(lk, [&] { return ev->reached == ev->recorded; });
    return model::fails() ? hipErrorInvalidValue : hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    model::events--;
    return hipSuccess;
}

// ---- graphs: a graph is the number of steps captured ----
typedef int* hipGraph_t;
typedef int* hipGraphExec_t;
namespace model {
inline std::atomic<long> execs{0}, graphs{0}, steps_run{0};
}
inline hipError_t hipStreamBeginCapture(hipStream_t st, int) {
    if (model::fails()) return hipErrorInvalidValue;
    S(st)->capturing = true;
    S(st)->captured = 0;
    return hipSuccess;
}
inline hipError_t hipStreamEndCapture(hipStream_t st, hipGraph_t* g) {
    S(st)->capturing = false;
    if (model::fails()) return hipErrorInvalidValue;
    *g = new int(S(st)->captured);
    model::graphs++;
    return hipSuccess;
}
inline hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, void*, void*, size_t) {
    if (model::fails()) return hipErrorOutOfMemory;
    *e = new int(*g);
    model::execs++;
    return hipSuccess;
}
inline hipError_t hipGraphDestroy(hipGraph_t g) {
    delete g;
    model::graphs--;
    return hipSuccess;
}
inline hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    delete e;
    model::execs--;
    return hipSuccess;
}
inline hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    if (model::fails()) return hipErrorInvalidValue;
    model::steps_run += *e;
    return hipSuccess;
}
