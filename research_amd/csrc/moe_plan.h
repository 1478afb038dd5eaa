// Host-testable arithmetic of the expert products: how many tiles the lists can make and which kernel runs them.  Plain C++.
#pragma once
#include <stdint.h>

// Tiles of `bm` items that `items` items of at most `experts` lists can make: every list leaves one tile part-filled, and
// no more lists than items are non-empty.
static inline int64_t moe_max_tiles(int64_t items, int experts, int bm) {
    const int64_t lists = items < experts ? items : experts;
    return lists + (items - lists) / bm;
}

enum MoeShape { kMoeStream, kMoeTile64, kMoeTile256 };

// By the items an expert has on average (lists of unequal length fill the next tile up).
static inline MoeShape moe_shape(int64_t items, int experts) {
    const int64_t mean = items / experts;
    return mean <= 4 ? kMoeStream : mean <= 8 ? kMoeTile64 : kMoeTile256;
}

// Whether tiles of 256 items, n_tiles over the outputs, are the faster ones for kMoeTile256.  They read an expert's weights once where
// tiles of 64 read them for each, and leave out what an empty part of a tile would multiply, but there have to be enough of them
// for the compute units: two thirds of one each, more than two of few items (of which the last round may be nearly empty).
// us, tiles of 64 -> of 256: 64 experts of 4096 x 1408 (704 and 1024 tiles): 10 items 493 -> 479, 25 items 575 -> 500, 125 items
// 1040 -> 568; of 2048 x 768 (384 and 512): 12 items 173 -> 189, 28 items 203 -> 197; 16 experts of 2048 x 768 (96 and 128):
// 37 items 79 -> 86, 112 items 87 -> 89.
static inline bool moe_stays(int64_t items, int experts, int64_t n_tiles, int cus) {
    const int64_t mean = items / experts, tiles = (items < experts ? items : experts) * n_tiles;
    return mean > 160 || tiles > 2 * (int64_t)cus || (mean > 24 && 3 * tiles >= 2 * (int64_t)cus);
}

// Rows of a part of the choice of experts (one workgroup): few parts, so that a part's place behind the others is quickly
// summed, but one row per wave (sixteen per workgroup) while there are few rows; a part's items fit LDS.
static inline int moe_part_rows(int64_t rows, int top) {
    int64_t n = (rows + 255) / 256;
    if (n < 16) n = 16;
    const int64_t most = 8192 / top;
    return (int)(n < most ? n : most);
}
static inline int64_t moe_parts(int64_t rows, int top) { return (rows + moe_part_rows(rows, top) - 1) / moe_part_rows(rows, top); }
