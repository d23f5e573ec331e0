// s2x_plan.h -- the rules by which the launchers choose grids and operand
// layouts from sizes (internal; host code only, no HIP types, so that the
// CPU tests compile it as it is).
#pragma once

#include <stdint.h>

namespace s2x {

// Most threads of a launch along x (HIP refuses a grid of 2^32 and more).
constexpr int64_t GRID_MAX_THREADS = 0xffffffffll;

// The grid of one operand of k_f16_operands: rows of ld halves, a thread per
// 8 of them, in blocks of 256.  A row has as many lanes as its chunks of 8
// need (a power of two, at most the 64 of a wave, then 512 columns a block),
// so that narrow rows share a wave.  64 lanes for any row leave 60 of them
// idle at 32 halves: 1,000,000 rows of K = 8 took 193 us with their GEMM of N =
// 16, now 74.
struct F16OperandGrid {
    int     lg_lanes;    // log2 of the lanes per row
    int64_t col_blocks;  // blocks per row group
    int64_t blocks;
};
inline F16OperandGrid f16_operand_grid(int64_t rows, int64_t ld) {
    F16OperandGrid g{0, 0, 0};
    const int64_t chunks = ld / 8;
    while (g.lg_lanes < 6 && (1ll << g.lg_lanes) < chunks) ++g.lg_lanes;
    const int64_t rows_per_block = 256 >> g.lg_lanes;
    g.col_blocks = (chunks + (1ll << g.lg_lanes) - 1) >> g.lg_lanes;
    g.blocks = (rows + rows_per_block - 1) / rows_per_block * g.col_blocks;
    return g;
}

}  // namespace s2x
