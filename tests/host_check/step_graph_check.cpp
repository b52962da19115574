// Replayed steps against the model of the runtime: the steps run are the
// steps asked for, the stream of the run is never the one captured (another
// thread may wait for it at any time, and does here), and after a call that
// fails the next run is whole and nothing is left over.
#include <cstdio>

#include "model_pool.h"
#include "dg_step_graph.h"

using namespace dgmi;

int main() {
    hipStream_t run = nullptr;
    CHECK(pool_stream(&run));
    std::atomic<bool> over{false};
    std::atomic<long> bad_waits{0};
    std::thread waiter([&] {
        while (!over) {
            if (S(run)->capturing) bad_waits++;
            std::this_thread::yield();
        }
    });
    const auto enqueue = [&](int k, hipStream_t on) {
        CHECK(S(on)->capturing && S(on)->device == S(run)->device);
        S(on)->captured += k;
        return Status::ok();
    };
    {
        StepGraph g;
        long want = 0;
        for (int n : {1, 0, 7, 8, 3, 40, 5, 200, 64, 1}) {
            CHECK(g.run(run, n, enqueue));
            CHECK(model::steps_run == (want += n));
        }
        CHECK(model::execs == 2);
        g.drop();
        CHECK(model::execs == 0);
    }
    for (long at = 0; at < 40; at++) {  // every call fails once
        StepGraph g;
        model::steps_run = 0;
        model::calls = 0;
        model::fail_at = at;
        const bool ok = (bool)g.run(run, 64, enqueue);
        const bool reached = model::calls > at;
        model::fail_at = -1;
        CHECK(ok == !reached);
        model::steps_run = 0;
        CHECK(g.run(run, 17, enqueue) && model::steps_run == 17);
        g.drop();
        CHECK(model::execs == 0 && model::graphs == 0);
        if (!reached) break;
        CHECK(at < 39);
    }
    {
        StepGraph g;  // a step that cannot be put on the stream
        CHECK(!g.run(run, 4, [](int, hipStream_t) { return Status::err(DG_ERR_ARG, "no"); }));
        CHECK(model::graphs == 0 && model::execs == 0);
    }
    {
        StepGraph g;  // with another device current
        model::device = 1;
        CHECK(g.run(run, 40, enqueue) && model::device == 1);
        model::device = 0;
    }
    over = true;
    waiter.join();
    CHECK(bad_waits == 0);
    pool_release_stream(run);
    CHECK(stream_pool().idle() == stream_pool().all.size());
    for (int d = 0; d < 2; d++)
        for (hipStream_t st : stream_pool().idle_of[d]) CHECK(S(st)->device == d);
    std::printf("step graphs ok\n");
    return 0;
}
