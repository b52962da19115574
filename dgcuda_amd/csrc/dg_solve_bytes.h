// Device bytes of a served solve (plain C++, checked on the CPU).
#pragma once
#include <cstdint>

#include "dg_device.h"

namespace dgmi {

// A request's size against the budget at submit, as stated in the interface:
// the FP64 tile layout counted with 16 mode slots.
inline int64_t estimate_bytes(int K, int N, int p, bool fp64) {
    const int64_t Kp = (K + 63) / 64 * 64;
    const int64_t s = fp64 ? 8 : 4;
    // p <= 4 reserves the matrix-core tile layout
    const bool tl = p >= 1 && p <= 4;
    const int64_t np = !tl ? n_modes(p) : !fp64 ? 4 * tile_groups(n_modes(p)) : 16;
    const int64_t ntiles = (K + 63) / 64;
    // matrix-core tiles (p >= 3 in a batch): packed geometry, 16 values per element
    const int64_t packed = p >= 3 ? 16 * s : 0;
    return Kp * (4 * N * np * s + 14 * s + 3 * 4 + 6 * 8 + 8 + 8 + 3 * 2 + packed) + ntiles * 64 * 4 + 4096;
}

// Device bytes a resident solve holds (the solver's allocations): the state
// arrays with the slots they have, the packed geometry of the Euler lane
// kernel (p <= 2 in a batch) where a tile's is not there, and the control
// block with its wave-speed slots.
inline int64_t held_bytes(int K, int N, int p, bool fp64) {
    const int64_t Kp = (K + 63) / 64 * 64;
    int64_t b = estimate_bytes(K, N, p, fp64);
    if (fp64) b -= Kp * 4 * N * (16 - tile64_slots(n_modes(p))) * 8;
    if (N == 4 && p <= 2) b += Kp * 16 * (fp64 ? 8 : 4);
    return b + (int64_t)CTRL_BYTES;
}

}  // namespace dgmi
