// Which part of the packed matrix a workgroup of the GEMV kernels takes.
#ifndef KX_TILE_ORDER_H
#define KX_TILE_ORDER_H

#include "kx_common.h"

namespace kx {

constexpr int kTileCols = 256;  // output columns per column tile: 128 bytes of a packed row
constexpr int kTileGroup = 8;   // most column tiles whose workgroups start side by side when they finish together

// The widest such group that divides the column tiles: no workgroup without a tile, no test for one.
inline int tile_group(int coltiles) {
    int side = kTileGroup;
    while (coltiles % side != 0) side--;
    return side;
}

// Which tile of a (column tiles x K tiles) grid a workgroup takes when neighbouring column tiles are to run on one XCD.
// Workgroups go to the eight XCDs in turn; the tiles, counted in groups of kTilesSideBySide columns with the columns of a
// group fastest, are cut into eight runs, one per XCD.  (One group of all columns would give an XCD few K tiles of many
// columns, and where the workgroup that comes last finishes a column alone, the XCD that is last would finish them all:
// 1024 -> 17704, groups of 32, M = 16 12.9 -> 17.0 us; groups of eight columns have a boundary more often, 15872 -> 18064 at
// M = 1 38.8 -> 40.4.)
struct TileOrder {
    uint32_t run = 0;          // tiles per XCD, 0: a workgroup takes the tile of its own number
    uint32_t extra = 0;        // the first `extra` XCDs take one more
    uint32_t whole = 0;        // columns in whole groups
    uint32_t in_whole = 0;     // tiles of those
    uint32_t group_magic = 0;  // divides by the tiles of a group
    uint32_t rest = 0;         // columns behind the whole groups
    uint32_t rest_magic = 0;   // divides by them; 0 for none and one
};
constexpr uint32_t kXcds = 8;
constexpr uint32_t kTilesSideBySide = 32;

// n / divisor = n * magic >> 32 where n * divisor < 2^32; divisor > 1
inline uint32_t magic_of(uint32_t divisor) {
    return static_cast<uint32_t>(((1ull << 32) + divisor - 1) / divisor);
}
__host__ __device__ inline uint32_t divide_by_magic(uint32_t n, uint32_t magic) {
    return static_cast<uint32_t>((static_cast<uint64_t>(n) * magic) >> 32);
}

inline TileOrder tile_order_of(uint32_t coltiles, uint32_t ktiles) {
    TileOrder o;
    const uint64_t tiles = static_cast<uint64_t>(coltiles) * ktiles, group = static_cast<uint64_t>(kTilesSideBySide) * ktiles;
    if (coltiles < 2 || tiles < 2 * kXcds || (tiles * group) >> 32) return o;
    o.run = static_cast<uint32_t>(tiles / kXcds);
    o.extra = static_cast<uint32_t>(tiles % kXcds);
    o.rest = coltiles % kTilesSideBySide;
    o.whole = coltiles - o.rest;
    o.in_whole = o.whole * ktiles;
    o.group_magic = magic_of(static_cast<uint32_t>(group));
    o.rest_magic = o.rest > 1 ? magic_of(o.rest) : 0u;
    return o;
}

struct Tile {
    int ct, kt;
};
// `id` counts the workgroups of the grid as they are dispatched.
__host__ __device__ __forceinline__ Tile tile_of_workgroup(const TileOrder& o, uint32_t id, uint32_t ktiles) {
    const uint32_t xcd = id % kXcds;
    uint32_t tile = xcd * o.run + (xcd < o.extra ? xcd : o.extra) + id / kXcds;
    if (tile < o.in_whole) {
        const uint32_t group = divide_by_magic(tile, o.group_magic);
        tile -= group * ktiles * kTilesSideBySide;
        return {static_cast<int>(group * kTilesSideBySide + tile % kTilesSideBySide), static_cast<int>(tile / kTilesSideBySide)};
    }
    tile -= o.in_whole;
    const uint32_t kt = o.rest_magic ? divide_by_magic(tile, o.rest_magic) : tile;
    return {static_cast<int>(o.whole + tile - kt * o.rest), static_cast<int>(kt)};
}

// Neighbouring column tiles share a memory line in every row whose 128-byte pieces do not start on a line: in the order of the
// numbers they lie on different XCDs, each of which fetches the line into its own L2.  us per launch at M = 1 / 2 / 4 / 8 / 16, by
// number -> by XCD: 4480 -> 20328 21.5 / 22.0 / 23.7 / 28.1 / 28.1 -> 15.6 / 17.3 / 18.6 / 23.4 / 23.9, 5472 -> 9000 with groups of 32
// 12.4 / 14.7 / 16.0 / 16.7 / 17.9 -> 10.1 / 13.5 / 13.3 / 13.9 / 15.5, 15872 -> 18064 with groups of 64 49.4 / 51.4 / 54.1 / 60.7 / 70.2 ->
// 38.8 / 41.8 / 43.3 / 50.3 / 61.5, 2176 -> 17792 (half a line) 8.3 / 10.0 / 11.0 / 12.8 / 14.9 -> 7.6 / 9.0 / 10.0 / 12.0 / 13.9.
// Where the pieces are whole lines nothing is shared, and neighbours on different XCDs are up to 15 % faster: 4096 -> 24576
// 13.9 / 15.3 / 16.6 / 19.3 / 20.3 by number against 14.6 / 15.8 / 17.7 / 21.1 / 21.2.
inline TileOrder packed_tile_order(const void* qweight, int N, int coltiles, int ktiles) {
    const bool whole_lines = N % kTileCols == 0 && reinterpret_cast<uintptr_t>(qweight) % 128 == 0;
    return whole_lines ? TileOrder{} : tile_order_of(static_cast<uint32_t>(coltiles), static_cast<uint32_t>(ktiles));
}

// Whether workgroups that finish a column tile together (`steps` 32-row steps for each of four waves and one block of K each) keep
// the order of the numbers all the same.  With a multiple of eight column tiles that order has every column on one XCD, and so the
// exchange, which grows with the rows, while the shared lines grow with the rows of W that a workgroup reads.  us per launch, by
// number -> by XCD, M = 16: one step 1024 -> 6072 7.6 -> 8.5, 2048 -> 4056 8.5 -> 9.4; two steps 5312 -> 1920 with groups of 64 behind
// SwiGLU 9.05 -> 10.2, 2048 -> 8168 9.3 -> 9.8; four steps 6144 -> 4056 (192 workgroups) 10.9 -> 11.3, 4096 -> 8168 (256) 12.6 -> 11.8;
// M = 9: one step 1024 -> 6072 7.25 -> 7.75, two 2048 -> 6072 8.3 -> 8.4, 2048 -> 8168 8.9 -> 8.9, four 4096 -> 6072 (192) 10.5 -> 10.2;
// M = 6: one step 1024 -> 8168 7.1 -> 7.4, two 2048 -> 8168 8.3 -> 8.2.
// With two and four column tiles an XCD's run is few rows of tiles and, unless the K tiles divide by eight, begins inside one:
// 6144 -> 264 (12 K tiles) at M = 6 / 16 8.3 / 8.8 -> 8.6 / 9.2, 2112 -> 896 with groups of 64 behind SwiGLU at M = 12 (9) 7.65 -> 8.0;
// 4096 -> 776 (16) at M = 6 / 16 7.5 / 8.1 -> 7.3 / 8.0.
// Where every other row starts on a line, half as many lines are shared, which four column tiles do not make up for: 2048 -> 896 with
// groups of 64 (eight) at M = 6 / 16 6.40 / 6.97 -> 6.64 / 7.21, 6144 -> 896 (24) at M = 9 / 16 8.41 / 8.56 -> 8.83 / 9.00; left out 12288 ->
// 896 (24, with groups of 64 48) at M = 6 9.46 -> 9.06 (9.69 -> 9.02) and at M = 9 with groups of 64 10.36 -> 9.98 (at M = 16 10.9 -> 12.0).
// More column tiles on such half lines lose by it as long as there is at most one workgroup per compute unit and few K tiles for the rows,
// those in groups of eight most, those in other even groups, whose columns lie on two or four XCDs, with one and two steps; odd groups
// have a column on all XCDs either way.  Groups of eight, four steps 15232 -> 1920 (240 workgroups, 30 K tiles) behind SwiGLU at M = 16
// 12.8 -> 13.4, 7680 -> 3968 (240, 15) at M = 15 11.8 -> 12.2; two 3328 -> 3968 (208, 13) at M = 7 7.8 -> 8.2, 1792 -> 8064 (224, 7)
// behind a norm at M = 8 7.6 -> 8.0; left out 14592 -> 1920 (232, 29) at M = 11 0.98 of the time, 4352 -> 3968 (272, 17) at M = 5 0.92.  Groups
// of six 3968 -> 2944 (192, 16) behind a norm at M = 10 8.8 -> 9.2, 3328 -> 1408 (78, 13) behind SwiGLU at M = 11 8.2 -> 8.4; left out
// 5632 -> 1408 (132, 22) at M = 7 0.95, 2048 -> 13696 (432, 8) at M = 10 0.985, four steps 1.00 up to K tiles for 2 M, then 0.95.
inline bool together_by_number(int M, int steps, int N, int coltiles, int ktiles) {
    const int workgroups = coltiles * ktiles, side = tile_group(coltiles);
    const bool half_lines = N % kTileCols == kTileCols / 2;
    if (half_lines && workgroups <= 256 && coltiles > 4) {
        if (side == static_cast<int>(kXcds) && (steps == 4 ? 5 * ktiles <= 12 * M : ktiles <= 3 * M)) return true;
        if (side % 2 == 0 && steps <= 2 && ktiles <= 2 * M) return true;
    }
    if (coltiles % static_cast<int>(kXcds) == 0) return 4 * steps < M || workgroups <= 12 * M;
    if (coltiles == 4 && half_lines && (M > 12 || ktiles <= (M > 8 ? 24 : 16))) return true;
    return (coltiles == 2 || coltiles == 4) && ktiles % static_cast<int>(kXcds) != 0;
}

// The same where one workgroup reads a column tile back and the grid, two workgroups to a compute unit, comes in rounds (four steps
// per wave, five rows and more).  Where the XCDs' runs begin on the same columns, as they do with a multiple of eight K tiles, or the last
// round is all but empty, the columns that are left for the end are the same on every XCD.  us per launch, by number -> by XCD, groups
// of 64 and 32: 22464 -> 2944 (528 workgroups, 44 K tiles) at M = 16 31.6 -> 38.5, 16256 -> 4736 (608, 32) at M = 10 27.2 -> 31.0, 20480 -> 3712
// (600, 40) behind SwiGLU at M = 10 32.5 -> 38.4, 24128 -> 6016 (1152, 48) at M = 16 42.3 -> 47.3, 24448 -> 2944 (576, 48) at M = 8 23.6 ->
// 25.7.  What the rule leaves out, time by XCD over by number: past 544 workgroups at nine and more rows, other numbers of K tiles 0.93 to
// 1.04, more column tiles than lie side by side 0.92 to 1.06, 0.96 on average; up to eight rows 0.92 to 1.05, 0.95.
inline bool alone_by_number(int M, int steps, int coltiles, int ktiles) {
    const int workgroups = coltiles * ktiles;
    if (M < 5 || steps != 4 || workgroups <= 512) return false;
    if (M < 9) return ktiles > 32 && ktiles % 4 == 0 && workgroups <= 608;
    return workgroups <= 544 || (ktiles % static_cast<int>(kXcds) == 0 && coltiles <= static_cast<int>(kTilesSideBySide));
}

}  // namespace kx

#endif  // KX_TILE_ORDER_H
