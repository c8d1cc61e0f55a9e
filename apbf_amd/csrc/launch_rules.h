// Launch choices by list sizes, as plain host functions. Every choice computes
// the same results.
#pragma once
#include <cstdint>

namespace apbf {

// Lanes per particle of the neighbour walk for about n particles, whose mean
// neighbour row has 48 entries or more (long_rows). Fewer lanes per particle make
// larger groups, which share more of the walk, until too few waves are left (ms per
// walk at 4, 8, 16, 64 lanes: drop of 228 k particles 0.33, 0.35, 0.51, 1.0; of 101 k
// 0.208, 0.218, 0.275, 0.52; of 43 k 0.144, 0.104, 0.117, 0.196; pool of 7.9 M 1.83,
// 2.16, -, 5.8; of 262 k 0.108, 0.107, 0.131, 0.249; of 110 k 0.092, 0.083, 0.084,
// 0.134; of 33 k 0.048, 0.034, 0.030, 0.041; of 16 k 0.047, 0.030, 0.024, 0.024; of
// 1.7 k 0.043, 0.028, 0.022, 0.012). Where rows are long, particles of unlike widths
// meet in a group, and the widest one's box costs all: the drop of 1.1 M particles
// takes 1.46 ms with 4 and 1.53 with 8 lanes in its first substeps, but 2.25 and
// 1.93 (16: 2.13) over the 60 of its impact. Hence 8 from rows of 48 entries on; the
// pool of 8 M has rows of 26.
inline int walk_lanes_for(uint32_t n, bool long_rows) {
    if (n >= 131072u) return long_rows ? 8 : 4;
    return n >= 40960u ? 8 : n >= 8192u ? 16 : 64;
}
// Whether the solver's blocks take one row group per flush of their shift table
// instead of four. Where the rows leave the chip idle at the 64 or 128 rows that
// four groups are, one is faster (us per iteration at one, two and four groups: drop
// of 43 k particles 34, 38, 48; of 8 k 16, 22, 33; pool of 16 k 16, 20, 29; dam break
// of 110 k at 8 lanes 52, 55, 57); from 128 K rows on, fewer flushes win.
inline bool solve_few_rows(uint32_t n) { return n < 131072u; }
// Digit width and passes of a sort of up to `cap` keys with the given digit width
// (shape_bits: 4, 8 or 11). keys_below: every key is below upper_bound; otherwise the
// keys are sorted by the whole digits that cover upper_bound.
//  * Up to SORT_SMALL values and 8-bit digits, all passes run in one launch of one
//    block (one_block); a list beyond 4 096 would leave the chip to one CU for longer
//    than the launches take that it saves. Against the two launches of each 9-bit
//    pass, in us per substep: 18-bit keys, 1 728 and 4 096 particles 106.0 and 108.4,
//    against 109.0 and 112.7; 9-bit keys, 729 particles 81.9 against 83.9, but 1 728,
//    3 375 and 4 096 particles 89.6, 95.9, 98.7 against 88.8, 95.3, 98.0. Hence two
//    launches for a single 9-bit pass over more than 1 024 values (SORT_SINGLE).
//  * Keys known to lie below the bound need the bits of bound - 1 only (a cell count
//    is a power of two: one bit less), and 9-bit digits where they save a pass of the
//    default 8 (18 bits: two passes instead of three).
constexpr uint32_t SORT_SMALL = 4096, SORT_SINGLE = 1024;
struct SortPlan {
    uint32_t bits, passes;
    bool one_block;
};
inline SortPlan sort_plan(uint32_t cap, uint32_t upper_bound, uint32_t shape_bits, bool keys_below) {
    if (keys_below && upper_bound) --upper_bound;
    uint32_t key_bits = 0;
    while (key_bits < 32u && (upper_bound >> key_bits) != 0u) ++key_bits;
    const uint32_t passes = (key_bits + shape_bits - 1u) / shape_bits, nines = (key_bits + 8u) / 9u;
    const bool nine = shape_bits == 8u && keys_below && nines < passes;
    const bool one_block = shape_bits == 8u && cap <= SORT_SMALL && !(nine && nines == 1u && cap > SORT_SINGLE);
    return nine && !one_block ? SortPlan{9u, nines, false} : SortPlan{shape_bits, passes, one_block};
}
// The walk's lane counts and those of the solver, all of them tried by the autotuner.
constexpr int WALK_LANES[] = {4, 8, 16, 64};
constexpr int SOLVE_LANES[] = {8, 16, 32};

}  // namespace apbf
