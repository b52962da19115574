// The streams and statuses that the checked host code takes from the solver.
#pragma once
#include "dg_solver.h"

namespace dgmi {

struct StreamPool {
    std::mutex mu;
    std::vector<std::unique_ptr<model::Stream>> all;
    std::vector<hipStream_t> idle;
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
    if (P.idle.empty()) {
        P.all.emplace_back(new model::Stream());
        P.idle.push_back(P.all.back().get());
    }
    *s = P.idle.back();
    P.idle.pop_back();
    return Status::ok();
}
void pool_release_stream(hipStream_t s) {
    if (!s) return;
    StreamPool& P = stream_pool();
    std::lock_guard<std::mutex> lk(P.mu);
    P.idle.push_back(s);
}

}  // namespace dgmi

#define CHECK(x)                                                  \
    do {                                                          \
        if (!(x)) {                                               \
            std::printf("FAIL line %d: %s\n", __LINE__, #x);      \
            std::exit(1);                                         \
        }                                                         \
    } while (0)
