// Output tile of a grouped forward or dgrad launch of more than 300 ring tiles on K-step-major operands (the smaller ones are priced
// in mx_gemm.hip).  Host arithmetic only.
//
// Such a launch is bound by reading the weights.  Up to 192 MiB of codes that this very call has quantised come out of the memory-side
// cache, and what counts is how soon a workgroup is through: 64 x 64 tiles up to 32 rows per group, 128 x 128 up to 192.  Larger ones,
// and copies that a caller has kept, come from memory (between two passes over a layer a model reads all the others), which the ring
// kernel reads best; with few rows, and short contractions, its rounds of mostly empty tiles cost more than small tiles' reads.
// dgrad's transposed codes are the forward's, which may be long ago: 128 x 128 tiles up to 192 rows are level there at worst.  E2M1
// weights against FP8 rows are half the bytes, which shifts the lines up.
//
// us of a launch, 64 x 64 / 64 x 128 / 128 x 128 / ring, groups of uneven size, its operands in the cache (launched again), behind the
// quantiser (codes streamed past the caches), and cold:
//   64 groups, [2816, 1024], 32 rows per group 33 / 35 / 35 / 46, 48 / 44 / 48 / 50, 74 / 74 / 74 / 74;
//     64 rows 39 / 42 / 40 / 47, 55 / 53 / 49 / 53, 81 / 78 / 77 / 76; 192 rows 75 / 71 / 56 / 62, 105 / 95 / 76 / 73, 132 / 118 / 98 / 93
//   the same with transposed codes, 64 x 128 / 128 x 128 / ring, in the cache and cold: 64 rows 43 / 40 / 50, 77 / 75 / 87; 192 rows
//     73 / 57 / 65, 116 / 98 / 101
//   E2M1, 16 groups, [14336, 1536], 32 rows 33 / 37 / 37 / 46, 48 / 47 / 50 / 51, 73 / 74 / 76 / 73; 192 rows 83 / 78 / 60 / 65,
//     114 / 103 / 83 / 71, 141 / 125 / 106 / 88
//   64 groups, [6144, 3584], 16 rows 312 / 283 / 299 / 264 behind the quantiser, 339 / 319 / 330 / 303 cold; 64 rows 383 / 352 / 317 / 264
//   E2M1 weights, FP8 rows, 64 groups, [2816, 2048], 64 rows 58 / 43 / 46 / 52, 82 / 57 / 61 / 59, 110 / 83 / 84 / 80; 128 rows
//     90 / 58 / 59 / 68, 125 / 79 / 76 / 69, 162 / 104 / 99 / 90; 128 groups, [5760, 2880], 48 rows, cold, 448 / 329 / 335 / 304
// The forward in two calls, the rule for fresh codes and the one for codes from memory, us: 32 groups, [4096, 1024], 48, 96, 192 rows
// 97 / 104, 104 / 106, 117 / 131; E2M1, 64 groups, [2048, 1408], 48, 192 rows 108 / 114, 134 / 137; E2M1 weights, FP8 rows, 64 groups,
// [2816, 2048], 96 and 128 rows 230 / 241, 245 / 250.  Tensor-wise, whose codes are streamed but whose weights have just been read
// twice, forward and backward, 64 groups, [2048, 1408], 64 rows 350 / 356.  Four layers forward and then backward, which gives dgrad cold
// codes: FP8, 64 groups, [2048, 1408], 160 rows 382 with 128 x 128 tiles up to 192 rows, 389 up to 128.
// The forward on eight kept copies in turn, tiles as for fresh codes / as from memory, on two cards, of which one runs the ring kernel
// up to 15 % slower than the other and the small tiles alike (hence no ring below 65 rows): FP8, 64 groups, [2816, 1024], 32 rows
// 52.5 / 46.5 and 52.1 / 46.6, 192 rows 86.7 / 83.1 and 87.3 / 90.5; [2048, 1408], 128 rows 67.9 / 63.1 and 68.1 / 65.0; E2M1, 16 groups,
// [14336, 1536], 32 rows 49.5 / 47.1 and 49.5 / 47.0, 160 rows 83.0 / 68.4 and 83.0 / 75.7 (64 rows on ring tiles 55 / 54 and 55 / 62); E2M1
// weights, FP8 rows, 128 groups, [2816, 2048], 96 rows on ring tiles 145 / 136 and 145 / 147, 128 rows 175 / 154 and 174 / 162.
#pragma once
#include <stdint.h>

namespace mxl {

enum { TILE_RING = 0, TILE_64 = 1, TILE_64x128 = 2, TILE_128 = 3 };

// weight_bytes: of all groups' codes; rows: per group, on average; steps: K steps of the contraction (64 elements, E2M1 rows 128);
// fresh: the call that launches has quantised the weights itself
inline int grouped_tile(int64_t weight_bytes, int64_t rows, int64_t steps, bool act_e2m1, bool e2m1_weights, bool bt, bool fresh) {
    const bool small = weight_bytes <= (int64_t)192 << 20;
    fresh = fresh && small;
    if (e2m1_weights) return rows <= (steps >= 40 ? 32 : fresh ? 128 : 96) ? TILE_64x128 : TILE_RING;
    if (small && bt) return rows <= 192 ? TILE_128 : TILE_RING;
    if (fresh) return rows <= 32 ? TILE_64 : rows <= 192 ? TILE_128 : TILE_RING;
    if (small) return rows <= 32 ? TILE_64x128 : rows <= 64 ? TILE_128 : TILE_RING;
    if (rows <= 16) return TILE_64x128;
    if (rows <= 32) return bt || act_e2m1 || steps < 40 ? TILE_64x128 : TILE_RING;
    return bt && rows <= 64 ? TILE_128 : TILE_RING;
}

}  // namespace mxl
