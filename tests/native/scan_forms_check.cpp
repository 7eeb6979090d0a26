// Host replay of the choice between the device-wide scan's forms (test only, plain C++).
//
// For each element type and size given, the form that scan_layout chooses (single-wave tiles with
// one look-back, groups of small tiles, groups of large tiles) has to cover every element once, to
// stay within the slots and grid that its kernel has, and to fit the workspace sized by the small
// tiles. Prints "ok <checks>" or the first violation and exits 1.
#include <stdio.h>
#include <stdlib.h>
#include "scan_layout.hpp"

namespace sl = cdna4::scan_layout;

static unsigned long long g_checks = 0;
#define CHECK(cond, what)                                                             \
    do {                                                                              \
        ++g_checks;                                                                   \
        if (!(cond)) { printf("violation: %s: %s n %zu\n", what, T.name, n); exit(1); } \
    } while (0)

struct Type { const char* name; int in_bytes, VEC, NW; };
static const Type kTypes[] = {{"32-bit", 4, 4, 1}, {"64-bit", 8, 2, 2}, {"16-bit", 2, 4, 1}};

int main(int argc, char** argv) {
    for (const Type& T : kTypes)
        for (int a = 1; a < argc; ++a) {
            const size_t n = strtoull(argv[a], nullptr, 10);
            const size_t ws = sl::ws_bytes(sl::tiles_for(n, T.VEC, sl::scan_u(T.in_bytes, false)));
            const int u = sl::spread_u(n, T.VEC);
            if (u) {
                CHECK(u == 2 || u == 4 || u == 8 || u == sl::kSpreadMaxU, "a compiled tile size");
                const size_t tiles = sl::tiles_for(n, T.VEC, u), tile = sl::tile_elems(T.VEC, u);
                CHECK(tiles >= 1 && tiles <= (size_t)sl::kSpreadTiles, "one slot per lane and pass");
                CHECK((tiles - 1) * tile < n && n <= tiles * tile, "the tiles cover the input");
                CHECK(sl::agg_offset() + sl::slot_word(tiles - 1, T.NW, T.NW - 1) * 8 + 8 <= ws, "slots in the workspace");
                CHECK(!sl::large_tiles(n, T.VEC, T.in_bytes), "the forms do not overlap");
                continue;
            }
            if (T.in_bytes == 8) {   // one round of large groups and not two of small ones (256 CUs)
                const size_t small_g = sl::groups_for(sl::tiles_for(n, T.VEC, sl::scan_u(8, false)), sl::scan_waves(8));
                const size_t large_g = sl::groups_for(sl::tiles_for(n, T.VEC, sl::scan_u(8, true)), sl::scan_waves(8));
                CHECK(small_g <= 256 || large_g > 256 || sl::large_tiles(n, T.VEC, 8), "one round of groups");
            }
            for (int vec = 0; vec < 2; ++vec) {
                const bool large = sl::large_tiles(n, T.VEC, T.in_bytes), v = vec && large;
                const int U = sl::scan_u(T.in_bytes, large), waves = sl::scan_waves(T.in_bytes);
                const size_t m = sl::main_elems(n, v, T.VEC), tiles = sl::tiles_for(m, T.VEC, U), tile = sl::tile_elems(T.VEC, U);
                const size_t groups = sl::groups_for(tiles, waves);
                CHECK(groups > 1, "several groups");
                CHECK((tiles - 1) * tile < m && m <= tiles * tile && n - m < (size_t)T.VEC, "the tiles cover the input");
                CHECK(groups * waves >= tiles && (groups - 1) * waves < tiles, "the groups cover the tiles");
                CHECK(sl::agg_offset() + groups * T.NW * 8 <= sl::pre_offset(groups), "agg before pre");
                CHECK(sl::pre_offset(groups) + groups * T.NW * 8 <= sl::xchg_offset(groups), "pre before the lines");
                CHECK(sl::xchg_offset(groups) + groups * sl::kXchgStride <= ws, "lines in the workspace");
            }
        }
    printf("ok %llu\n", g_checks);
    return 0;
}
