// A step captured for replay, alone and MANY times in a row.
#pragma once
#include "dg_solver.h"

namespace dgmi {

// Between two graph launches the device idles about 7 us (it replays the
// kernels of one graph 3-5 us apart, launches included), so steps are
// replayed MANY to a graph: a step of advection p = 1 FP64 on 2,048 triangles
// 26.7 -> 20.2 us, Euler p = 2 FP32 32,768 40.1 -> 33.4, p = 1 FP32 500,000
// 91.8 -> 85.7, p = 4 FP32 524,288 385 -> 381 (4 to a graph: 21.1, 34.3, 86.2;
// 16: no further gain).  The long graph is captured once its steps repay it:
// from MANY_FROM steps on, counted since the last change of the step.
class StepGraph {
   public:
    static constexpr int MANY = 8;
    static constexpr int64_t MANY_FROM = 32;
    ~StepGraph() { drop(); }

    // the captured step is out of date
    void drop() {
        for (hipGraphExec_t* g : {&one, &many}) {
            if (*g) (void)hipGraphExecDestroy(*g);
            *g = nullptr;
        }
        taken = 0;
    }

    // `n` steps on stream `st`; `enqueue(k, on)` puts k steps on stream `on`
    template <typename F>
    Status run(hipStream_t st, int64_t n, F&& enqueue) {
        while (n > 0) {
            const bool long_graph = n >= MANY && (many || taken + n >= MANY_FROM);
            hipGraphExec_t& g = long_graph ? many : one;
            const int len = long_graph ? MANY : 1;
            if (!g) {
                Status s = capture(st, len, g, enqueue);
                if (!s) return s;
            }
            hipError_t e = hipGraphLaunch(g, st);
            if (e != hipSuccess) return hip_status(e, "step graph launch");
            n -= len;
            taken += len;
        }
        return Status::ok();
    }

   private:
    hipGraphExec_t one = nullptr, many = nullptr;
    int64_t taken = 0;

    // On a stream of its own, of the device of `run`: the solve's stream may be
    // in use meanwhile (a thread reading the state during a run; the long graph
    // is captured in the middle of one), and a wait for a stream that is being
    // captured fails.
    template <typename F>
    static Status capture(hipStream_t run, int len, hipGraphExec_t& out, F&& enqueue) {
        hipDevice_t dev = 0;
        hipError_t e = hipStreamGetDevice(run, &dev);
        if (e != hipSuccess) return hip_status(e, "step capture");
        const OnDevice here(dev);
        struct OwnStream {
            hipStream_t st = nullptr;
            ~OwnStream() { pool_release_stream(st); }
        } own;
        Status s = pool_stream(&own.st);
        if (!s) return s;
        e = hipStreamBeginCapture(own.st, hipStreamCaptureModeThreadLocal);
        if (e != hipSuccess) return hip_status(e, "step capture");
        s = enqueue(len, own.st);
        hipGraph_t gr = nullptr;
        e = hipStreamEndCapture(own.st, &gr);
        if (s && e == hipSuccess) e = hipGraphInstantiate(&out, gr, nullptr, nullptr, 0);
        if (gr) (void)hipGraphDestroy(gr);
        if (!s) return s;
        return hip_status(e, "step capture");
    }
};

}  // namespace dgmi
