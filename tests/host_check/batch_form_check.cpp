// The launch form an FP64 batch takes by itself (dg_worklist.h).
#include <cstdio>

#include "dg_worklist.h"

using namespace dgmi;

#define CHECK(x)                                             \
    do {                                                     \
        if (!(x)) {                                          \
            std::printf("FAIL line %d: %s\n", __LINE__, #x); \
            return 1;                                        \
        }                                                    \
    } while (0)

int main() {
    for (int64_t e : {int64_t(2), int64_t(2360), int64_t(524287), int64_t(5000000)})
        for (bool running : {false, true})
            for (bool now : {false, true}) {  // one class: nothing to gain from sharing a launch
                CHECK(take_per_class(1, 0, e, running, now));
                CHECK(take_per_class(0, 1, e, running, now));
            }
    const struct { int lanes, tiles; int64_t line; } lists[] = {{1, 1, 65536}, {0, 2, 65536}, {2, 0, 524288}, {2, 1, 524288},
                                                               {1, 2, 524288}, {2, 2, 524288}};
    for (const auto& l : lists) {
        CHECK(!take_per_class(l.lanes, l.tiles, l.line - 1, false, false));
        CHECK(take_per_class(l.lanes, l.tiles, l.line, false, false));
        // a list that runs keeps its form while its triangles move about the line
        int changes = 0;
        bool now = false;
        for (int i = 0; i < 100; i++) {
            const bool f = take_per_class(l.lanes, l.tiles, l.line + (i % 2 ? 1 : -1) * l.line / 10, true, now);
            changes += f != now;
            now = f;
        }
        CHECK(changes == 0);
        CHECK(take_per_class(l.lanes, l.tiles, l.line + l.line / 8, true, false));
        CHECK(!take_per_class(l.lanes, l.tiles, l.line - l.line / 8 - 1, true, true));
    }
    std::printf("batch form ok\n");
    return 0;
}
