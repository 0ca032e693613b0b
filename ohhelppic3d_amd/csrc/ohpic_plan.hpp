// ohpic_plan.hpp -- which tiles are split, and the order they are dispatched in.
//
// Plain C++ (no HIP): the host runtime of libohpic.so plans with it, and the
// CPU tests compile it alone.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace ohpic {

// One tile of one instance as plan_chunks sees it.
struct TileLoad {
    int inst, tile;
    int64_t load;  // bin slots over all species
};

// No chunk is made smaller than this many slots: it costs an E tile, a charge
// flush (tiles of 9.4K slots in 2 chunks: 32^3 x 64 ppc mixed 124 us per launch,
// whole 88 us).
constexpr int64_t kMinChunkLoad = 8192;

// Octave of a load in eighths: floor(8 log2 load), -1 for none.  (Whole
// numbers: the plan takes one per tile, and 2^(k/8) are no fractions of loads.)
inline int load_level(int64_t load)
{
    if (load <= 0) return -1;
    // 2^(63 + k/8), rounded down
    constexpr uint64_t kEighth[7] = {0x8b95c1e3ea8bd6e6u, 0x9837f0518db8a96fu, 0xa5fed6a9b15138eau,
                                     0xb504f333f9de6484u, 0xc5672a115506daddu, 0xd744fccad69d6af4u,
                                     0xeac0c6e7dd24392eu};
    const int lz = __builtin_clzll((uint64_t)load);
    const uint64_t m = (uint64_t)load << lz;
    int k = 0;
    while (k < 7 && m > kEighth[k]) ++k;
    return 8 * (63 - lz) + k;
}

// Sorts the tiles by load level, heaviest first, tiles of one level in the
// given order.  (By counting: a comparison sort that took the levels' logarithms
// as it compared cost 0.9 ms per plan of 2496 tiles and 13 ms of 32768, this
// 0.04 and 0.6.)
inline void sort_by_level(std::vector<TileLoad> &tiles)
{
    constexpr int kTop = 8 * 62 + 7;  // level of the largest load
    std::vector<int16_t> key(tiles.size());
    std::vector<size_t> at(kTop + 3, 0);
    for (size_t i = 0; i < tiles.size(); ++i) {
        key[i] = (int16_t)(kTop - load_level(tiles[i].load));
        ++at[key[i] + 1];
    }
    for (size_t k = 1; k < at.size(); ++k) at[k] += at[k - 1];
    std::vector<TileLoad> out(tiles.size());
    for (size_t i = 0; i < tiles.size(); ++i) out[at[key[i]]++] = tiles[i];
    tiles.swap(out);
}

// Chunks per tile (nch[i] of tiles[i]) and the order the tiles are dispatched
// in, for `slots` workgroups resident at once: heaviest first (in steps of an
// eighth of an octave, tiles of one step in grid order).  A tile stays whole
// unless it would outlast the launch: split are the tiles of a grid with less
// than a quarter as many tiles as workgroups, so that they fill the device
// (16^3 x 200 ppc: 169 -> 149 us mixed, 189 -> 158 us FP64; with half as many,
// 32^3 x 300 ppc mixed, whole tiles are faster, 317 against 363 us), and tiles
// at least twice as heavy as the mean that hold at least a workgroup's
// fair share of the work (a density peak).  Splitting further, so that the
// last tiles of a launch end together, costs more than it gives (80x72x88 x 20
// ppc mixed: 317 us per launch against 280).  At most max_extra items beyond
// one per tile.  A group is planned as one: 32 members of 16^3-64^3, each
// split as if it ran alone (62936 items), took 3.01 ms per particle launch,
// planned together (5472 items) 1.4 ms.
inline void plan_chunks(std::vector<TileLoad> &tiles, int64_t slots, int64_t max_extra,
                        std::vector<int> &nch)
{
    sort_by_level(tiles);
    nch.assign(tiles.size(), 1);
    if (tiles.empty()) return;
    int64_t work = 0, extra = 0;
    for (const TileLoad &t : tiles) work += t.load;
    const int64_t share = work / slots, nt = (int64_t)tiles.size();
    const int64_t unit = std::max(
        kMinChunkLoad, 4 * nt <= slots ? share : std::max(share / 2, work / nt));
    for (size_t i = 0; i < tiles.size(); ++i) {
        const int64_t want = tiles[i].load / unit;
        nch[i] = (int)std::max<int64_t>(1, std::min<int64_t>({want, 1 + max_extra - extra, 256}));
        extra += nch[i] - 1;
    }
}

}  // namespace ohpic
