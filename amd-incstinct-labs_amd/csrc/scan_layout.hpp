// Index and workspace arithmetic of the device-wide scan (reduce_scan.hip), as constexpr functions
// shared by the kernels, their launcher and a host-side replay (tests/native/scan_layout_check.cpp)
// that walks every load, store and tile-slot address of every tile for given sizes and checks it
// against the buffer and workspace sizes. Plain C++: clang compiles constexpr functions for host
// and device alike.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace cdna4 {
namespace scan_layout {

constexpr size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// A tile is 64 lanes x U vectors of VEC elements. U on the aligned path: kScanU for 4- and 8-byte
// inputs, twice that for 16-bit inputs (held packed, 8 bytes per vector); the small tiles of
// mid-size calls (vec false) half of kScanU.
constexpr int kScanU = 32;
constexpr int scan_u(int in_bytes, bool vec, int base = kScanU) { return vec ? (in_bytes == 2 ? 2 * base : base) : base / 2; }
constexpr size_t tile_elems(int vec, int u) { return (size_t)64 * vec * u; }
constexpr size_t tiles_for(size_t n, int vec, int u) { return (n + tile_elems(vec, u) - 1) / tile_elems(vec, u); }

// Workspace for `nslots` look-back slots (one per tile group): [error and epoch words, padded to 256 B]
// [agg slots: align256(nslots * 16)][pre slots: align256(nslots * 16)][exchange lines:
// nslots * kXchgStride], two 64-bit words per slot and array (one used by 32-bit values), and per
// group one 128-byte line in which its waves leave their tile totals and wave 0 the group's prefix
// (W + 1 values of at most 8 bytes, W the group's waves). The library sizes it by the small tiles'
// count, which bounds the group count of either size (and holds spread_u's slots: at two vectors a
// tile takes 16 bytes where a small tile of eight times its elements has 160).
constexpr size_t kXchgStride = 128;
constexpr size_t ws_bytes(size_t ntiles) { return 256 + 2 * align256(ntiles * 16) + align256(ntiles * kXchgStride); }
constexpr size_t agg_offset() { return 256; }
constexpr size_t pre_offset(size_t ntiles) { return 256 + align256(ntiles * 16); }
constexpr size_t xchg_offset(size_t ntiles) { return pre_offset(ntiles) + align256(ntiles * 16); }

// Aligned calls of large tiles scan whole VEC-element vectors in the tiles and the last n % VEC
// elements in a one-wave tail; all others scan every element in the tiles (vectors at any element,
// the last tile's incomplete vector element by element).
constexpr size_t main_elems(size_t n, bool vec, int VEC) { return vec ? n - n % (size_t)VEC : n; }

// Tile t starts at element t * TILE; the elements it covers (TILE, or fewer for the last tile).
constexpr size_t tile_base(size_t tile, size_t TILE) { return tile * TILE; }
constexpr bool tile_full(size_t base, size_t TILE, size_t n) { return base + TILE <= n; }
constexpr uint32_t tile_rem(size_t base, size_t TILE, size_t n) {
    return base + TILE <= n ? (uint32_t)TILE : (uint32_t)(n - base);
}
// Vector j of lane `lane` in a tile: its index among the tile's vectors, and the guard of the last
// (partial) tile: the vector is read and written only when it lies wholly inside the tile.
constexpr uint32_t vec_in_tile(int j, unsigned lane) { return (uint32_t)j * 64 + lane; }
constexpr bool vec_live(bool full, int j, unsigned lane, uint32_t rem, int VEC) {
    return full || vec_in_tile(j, lane) < rem / (uint32_t)VEC;
}
// Element e of vector j of a lane, for the elements that no whole vector holds.
constexpr uint32_t elem_in_tile(int j, unsigned lane, int e, int VEC) { return vec_in_tile(j, lane) * (uint32_t)VEC + e; }

// Tiles run in workgroups of W waves, one tile per wave: wave w of workgroup g scans tile g W + w
// (waves past the last tile load and store nothing). The waves' totals meet in the workgroup, and
// the look-back state (a slot per published value) is per workgroup: a group publishes the total
// of its tiles and then its inclusive prefix. W = 4, and 8 for 8-byte inputs, whose tiles hold
// half the elements of 4-byte ones, so that twice as many look-backs would trail the stream (i64
// 2^26: 199.8 us with four waves, 187.3 with eight; f32 100.8 with four, 112.6 with eight, 109.7
// with two; f16 77.5 / 83.1 / 87.2).
constexpr int kScanWavesMax = 8;
constexpr int scan_waves(int in_bytes) { return in_bytes == 8 ? 8 : 4; }
static_assert((kScanWavesMax + 1) * 8 <= (int)kXchgStride, "a group's exchange values fit its line");
constexpr size_t groups_for(size_t ntiles, int waves) { return (ntiles + waves - 1) / waves; }
constexpr size_t group_tile(size_t group, unsigned wave, int waves) { return group * waves + wave; }

// Which form scans n elements (times at f32, f16, i64 on the MI355X, us).
//
// Up to kSpreadTiles tiles of kSpreadMaxU vectors: single-wave tiles over the whole chip with one
// look-back over all of them (scan_spread). Vectors per lane: the fewest of 2, 4, 8 that need at
// most one tile per CU, then 8 and 16 with up to two (262,144 f32: 256 tiles 4.1, 512 tiles 5.1;
// 1,000,003 f32: 489 tiles of 8 vectors 6.9, 245 of 16 7.6). Against groups of large tiles:
// 1,000 elements 6.1 -> 3.5, 11.8 -> 3.6, 8.2 -> 4.1; 1,000,003 12.4 -> 7.1, 18.2 -> 7.0, 18.8 -> 9.0.
// No line by alignment: 16-bit inputs at elements 0 / 1 / 2 / 3 take 3.2 / 3.3 / 3.3 / 3.2 at 1,000, 6.7 /
// 6.4 / 6.7 / 6.9 at 1,000,000 and, in small tiles, 8.6 / 9.0 / 8.8 / 8.9 at 3,000,000.
constexpr int kSpreadTiles = 512;
constexpr int kSpreadMaxU = 16;
constexpr int spread_u(size_t n, int VEC) {
    constexpr size_t one = kSpreadTiles / 2;
    return tiles_for(n, VEC, 2) <= one ? 2
         : tiles_for(n, VEC, 4) <= one ? 4
         : tiles_for(n, VEC, 8) <= 2 * one ? 8
         : tiles_for(n, VEC, kSpreadMaxU) <= 2 * one ? kSpreadMaxU : 0;
}
// Above that large tiles from large_groups groups of them on, one and a half per CU, for 16-bit
// inputs, whose small tiles are a quarter, one; small tiles below. Fewer groups leave CUs idle
// (4,194,304 elements: 12.8 -> 10.2, 17.0 -> 9.1, 19.2 -> 14.9; 8,388,608: 17.7 -> 13.6, 18.2 ->
// 12.2, 23.0 -> 22.8; 12,000,000: 21.4 -> 18.8, 19.1 -> 16.1, 42.2 -> 38.3), more have fewer prefixes
// to wait for in large tiles (16,777,216 with the look-back in both: small 27.5, 24.3, 51.0, large
// 25.8, 20.4, 48.0).
constexpr int large_groups(int in_bytes) { return in_bytes == 2 ? 256 : 384; }
// 8-byte inputs also take them where small tiles need more than one group per CU and large ones do not
// (4.2 to 8.4 million elements): their groups are eight waves, and a second round of them waits for
// the first. Small / large, i64: 5,000,012 elements 19.4 / 18.2, 6,291,456 21.4 / 19.3, 8,388,608 24.7 /
// 22.8; vectors at odd elements 19.4 / 19.7, 21.9 / 20.6, 26.2 / 26.6.
constexpr size_t kOneRound = 256;
constexpr bool large_tiles(size_t n, int VEC, int in_bytes) {
    const size_t large = groups_for(tiles_for(n, VEC, scan_u(in_bytes, true)), scan_waves(in_bytes));
    const size_t small = groups_for(tiles_for(n, VEC, scan_u(in_bytes, false)), scan_waves(in_bytes));
    return large >= (size_t)large_groups(in_bytes) || (in_bytes == 8 && large <= kOneRound && small > kOneRound);
}

// 64-bit word w of group (slot) t's slot (NW words per slot).
constexpr size_t slot_word(size_t tile, int nw, unsigned w) { return tile * (size_t)nw + w; }

}  // namespace scan_layout
}  // namespace cdna4
