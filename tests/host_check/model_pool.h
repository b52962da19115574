// The streams and statuses that the checked host code takes from the solver.
#pragma once
#include "dg_solver.h"

namespace dgmi {

struct StreamPool {
    std::mutex mu;
    std::vector<std::unique_ptr<model::Stream>> all;
    std::vector<hipStream_t> idle_of[2];  // by device
    size_t idle() const { return idle_of[0].size() + idle_of[1].size(); }
};
inline StreamPool& stream_pool() {
    static StreamPool p;
    return p;
}
Status hip_status(hipError_t e, const char* what) {
    return e == hipSuccess ? Status::ok() : Status::err(DG_ERR_HIP, what);
}
Status pool_stream(hipStream_t* s) {
    if (model::fails()) return Status::err(DG_ERR_HIP, "stream");
    StreamPool& P = stream_pool();
    std::lock_guard<std::mutex> lk(P.mu);
    auto& idle = P.idle_of[model::device];
    if (idle.empty()) {
        P.all.emplace_back(new model::Stream());
        P.all.back()->device = model::device;
        idle.push_back(P.all.back().get());
    }
    *s = idle.back();
    idle.pop_back();
    return Status::ok();
}
void pool_release_stream(hipStream_t s) {
    if (!s) return;
    StreamPool& P = stream_pool();
    std::lock_guard<std::mutex> lk(P.mu);
    P.idle_of[model::device].push_back(s);
}

}  // namespace dgmi

#define CHECK(x)                                                  \
    do {                                                          \
        if (!(x)) {                                               \
            std::printf("FAIL line %d: %s\n", __LINE__, #x);      \
            std::exit(1);                                         \
        }                                                         \
    } while (0)
