// The bytes a served solve is counted with against its allocations, summed
// here array by array for the kernels a batch uses (lanes up to p = 2, tiles
// from p = 3, with the most sides and halo elements a tile can have).
#include <cstdio>

#include "dg_solve_bytes.h"

using namespace dgmi;

int main() {
    int bad = 0;
    for (int K : {2, 64, 66, 200, 1000, 8214, 100000, 524288})
        for (int N : {1, 4})
            for (int p = 1; p <= 4; p++)
                for (int fp64 = 0; fp64 < 2; fp64++) {
                    const int64_t Kp = (K + 63) / 64 * 64, s = fp64 ? 8 : 4, tiles = Kp / 64;
                    const StateIx ix{N, n_modes(p), (int)Kp, fp64 ? LAYOUT_TILE64 : LAYOUT_TILE32};
                    int64_t b = 4 * (int64_t)ix.elems() * s;       // c, acc, ua, ub
                    b += (5 + 9) * Kp * s + 3 * Kp * 4;            // geometry, neighbours
                    b += (6 + 1) * Kp * 8 + Kp * 4;                // vertices, Jacobian, order
                    b += (K + 255) / 256 * 8 * 8;                  // audit
                    b += (int64_t)CTRL_BYTES;
                    if (p >= 3) b += tiles * (4 + 64 * 4 + 192 * 4 * s) + 4 * Kp * s;  // counts, halo, sides, maps
                    if (p <= 2 && N == 4) b += 16 * Kp * s;        // the lane kernel's records
                    const int64_t held = held_bytes(K, N, p, fp64);
                    if (held < b || held > b + b / 4 + 16384) {
                        std::printf("FAIL K=%d N=%d p=%d fp64=%d: allocated %lld, counted %lld\n", K, N, p, fp64,
                                    (long long)b, (long long)held);
                        bad++;
                    }
                }
    if (!bad) std::printf("solve bytes ok\n");
    return bad != 0;
}
