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

// Row stride (halves) that the F16 GEMM takes: a tile's 128 rows within 31
// bits of bytes.
inline bool f16_ld_ok(int64_t ld) { return 128 * ld * 2 <= 0x7fffffff; }

// Operand layouts of one F16 product from raw weight rows (K halves apart)
// and a workspace of round_up(N K_pad 2, 256) + round_up(M K_pad 2, 256)
// bytes.  Weight rows that are 16-byte aligned (w_align16: their first one
// is) are read in place; X then has the whole workspace for rows of whole
// 128-byte lines, if those fit there and the GEMM takes the stride.
struct F16MulMatPlan {
    bool    w_direct;
    int64_t ldx16, ldw;  // halves
    int64_t x_off;       // bytes
    int64_t total;       // of the workspace
};
inline F16MulMatPlan f16_mul_mat_plan(int64_t K, int64_t N, int64_t M, bool w_align16) {
    const int64_t K_pad = (K + 31) / 32 * 32, ld_line = (K + 63) / 64 * 64;
    F16MulMatPlan p;
    p.x_off = (N * K_pad * 2 + 255) / 256 * 256;
    p.total = p.x_off + (M * K_pad * 2 + 255) / 256 * 256;
    p.w_direct = K % 8 == 0 && w_align16;
    p.ldw = p.w_direct ? K : K_pad;
    p.ldx16 = K_pad;
    if (p.w_direct && M * ld_line * 2 <= p.total && f16_ld_ok(ld_line)) {
        p.ldx16 = ld_line;
        p.x_off = 0;
    }
    return p;
}

}  // namespace s2x
