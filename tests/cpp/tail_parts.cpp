// K parts of a last round's tiles (host): lines of the rule for a lone round, at
// 32 CUs per XCD.
#include <cstdio>

#include "../../candle-moe_amd/csrc/cm_internal.hpp"

int main() {
    struct { int R, full, nk, want; } cases[] = {
        {2, 0, 32, 4}, {4, 0, 32, 4}, {8, 0, 32, 4}, {8, 0, 24, 3}, {6, 0, 24, 3}, {12, 0, 32, 2}, {4, 0, 64, 8},  // split
        {16, 0, 48, 2}, {1, 0, 64, 8},
        {8, 0, 16, 1}, {2, 0, 16, 1}, {16, 0, 24, 1}, {12, 0, 24, 1}, {16, 0, 32, 1}, {17, 0, 64, 1}, {0, 0, 64, 1},  // whole
        {8, 32, 16, 2}, {16, 32, 24, 2}, {16, 96, 32, 2}, {17, 32, 64, 1}, {4, 32, 15, 1},  // behind full rounds
    };
    int bad = 0;
    for (const auto& c : cases) {
        const int got = cm::tail_parts(c.R, 32, c.full, c.nk);
        if (got != c.want) {
            std::printf("R %d full %d K tiles %d: %d parts, expected %d\n", c.R, c.full, c.nk, got, c.want);
            bad = 1;
        }
    }
    if (!bad) std::printf("ok\n");
    return bad;
}
