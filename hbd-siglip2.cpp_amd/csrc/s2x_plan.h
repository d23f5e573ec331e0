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
// bytes.  Weight rows that are 16-byte aligned are read in place where neither
// y nor the workspace lies over them (f16_w_in_place); X then has the whole
// workspace for rows of whole 128-byte lines, if those fit there and the GEMM
// takes the stride.
struct F16MulMatPlan {
    bool    w_direct;
    int64_t ldx16, ldw;  // halves
    int64_t x_off;       // bytes
    int64_t total;       // of the workspace
};
inline F16MulMatPlan f16_mul_mat_plan(int64_t K, int64_t N, int64_t M, bool w_in_place) {
    const int64_t K_pad = (K + 31) / 32 * 32, ld_line = (K + 63) / 64 * 64;
    F16MulMatPlan p;
    p.x_off = (N * K_pad * 2 + 255) / 256 * 256;
    p.total = p.x_off + (M * K_pad * 2 + 255) / 256 * 256;
    p.w_direct = w_in_place;
    p.ldw = p.w_direct ? K : K_pad;
    p.ldx16 = K_pad;
    if (p.w_direct && M * ld_line * 2 <= p.total && f16_ld_ok(ld_line)) {
        p.ldx16 = ld_line;
        p.x_off = 0;
    }
    return p;
}

inline int64_t f16_mul_mat_ws_bytes(int64_t K, int64_t N, int64_t M) { return f16_mul_mat_plan(K, N, M, false).total; }
inline bool f16_w_in_place(uintptr_t w, uintptr_t y, uintptr_t ws, int64_t K, int64_t N, int64_t M) {
    const auto apart = [&](uintptr_t p, int64_t bytes) {
        return p + (uintptr_t)bytes <= w || w + (uintptr_t)(N * K * 2) <= p;
    };
    return K % 8 == 0 && w % 16 == 0 && apart(y, M * N * 4) && apart(ws, f16_mul_mat_ws_bytes(K, N, M));
}

// The tile form of an F16 product, by tiles per round of the 256 CUs (every
// form gives the same bits).  Small: 64 x 64 tiles, two workgroups a CU, while
// all of them are resident at once (M = 729, K = 4320, N = 1152: 18 us against
// 33 in 128 x 128 tiles; at 648 tiles, M = 729, K = 1152, N = 3456: 14.6
// against 12.4).  Above that 128 x 128 tiles, or 256 x 128 where that takes
// fewer rounds by more than the 1.6 x that a round of them is longer (and the
// taller tile's rows lie within 31 bits): M = 3645, K = 4320, N = 1152 (2
// rounds or 1) 63 against 51 us, M = 8640 (3 or 2) 103 against 107, M =
// 23,328 (7 or 4) 301 against 257.
enum class F16Form { Small, Mid, Wide };
inline F16Form f16_form(int64_t M, int64_t N, int64_t ldx) {
    const auto tiles = [&](int64_t bm, int64_t bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
    const auto rounds = [&](int64_t t) { return (t + 255) / 256; };
    if (tiles(64, 64) <= 512) return F16Form::Small;
    if (8 * rounds(tiles(256, 128)) < 5 * rounds(tiles(128, 128)) && 256 * ldx * 2 <= 0x7fffffff) return F16Form::Wide;
    return F16Form::Mid;
}

// The tile form of a tiled int8 product (s2x_gemm.hip).  Each output's K order
// is the same in all of them, so the choice does not change a bit.
enum class Q8Form {
    Wide,    // 128 x 128, the throughput form, two workgroups per CU
    Lone,    // latency forms of 32 x 32 waves: 32 x 32, one wave
    Narrow,  //   32 x 64, two waves
    Square,  //   64 x 64, four waves, two workgroups per CU
    Rows32,  //   32 x 128, four waves
    Small4,  // latency forms of 32 x 64 waves: 64 x 128, four stages, one workgroup per CU
    Small3   //   64 x 128, three stages, two workgroups per CU
};
// Wide for GEMMs of at least two 128 x 128 tiles per CU; below that the
// latency form (M = 729 in 128 x 128 tiles: out 19.8 us, fc2 58.7).  Near that
// line the two are within 8 % either way, by how full their last rounds are
// (K = 4320, N = 4304: M = 1800, 510 tiles, Small3 81.7 us, Wide 76.4; M =
// 2048, 544 tiles, 101.1 and 108.6).  The
// epilogues that work on 32 x 64 blocks (plain false: GELU -> Q8_1 / F16, QKV)
// have the 64 x 128 tiles, with four stages in the ring (three in flight)
// where their workgroups fit one per CU and three stages (two per CU)
// otherwise.  The plain / bias / residual ones (the out projection, fc2, the
// text tower's QKV) run the smallest tiles that still give every workgroup a
// CU of its own (a workgroup's DMA, about 40 bytes per ns from past the L2,
// is what a smaller tile shortens), then Square while all of them are
// resident: 16 KB of quants a stage where Rows32 takes 20.  Where Square is
// past one workgroup per CU, a few CUs have two and the others wait for them:
// Rows32 if that still is within one (K = 4320, N = 4304, M = 200: Rows32
// 18.2 us, Square 23.8, Narrow 23.7, Lone 25.9; K = 1152 7.7, 9.4, 9.4, 8.7).
// K = 4320, N = 1152: M = 64 Lone 16.4 us, Narrow 17.0, Square 17.5; M = 320
// Narrow 18.1 to 18.6, Lone 18.4, Square 18.7; M = 729 Square 20.2, Rows32
// 20.5, Narrow 25.3, Lone 33.4.  K = 1152: M = 320, N = 3456 Square 10.4,
// Narrow 13.9, Rows32 14.3; M = 1458, N = 1152 Square 11.6, Rows32 15.6.  More
// than two Square workgroups per CU: 64 x 128 tiles of waves with two
// subtiles (M = 1800: 43.1 us).
// A K split has n_split workgroups per tile, which count for what fits one per
// CU; Square and Wide end by the tiles of one range.  Counting those alone
// everywhere gave Narrow to K = 4320, N = 256, M = 1458 in 2 ranges: 17.7 us,
// Square 14.1.
inline Q8Form q8_form(int64_t M, int64_t N, bool plain, int64_t n_split = 1) {
    const auto grid = [&](int64_t bm, int64_t bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
    const auto tiles = [&](int64_t bm, int64_t bn) { return grid(bm, bn) * n_split; };
    if (grid(128, 128) >= 2 * 256) return Q8Form::Wide;
    if (!plain) return tiles(64, 128) <= 256 ? Q8Form::Small4 : Q8Form::Small3;
    if (tiles(32, 32) <= 256) return Q8Form::Lone;
    if (tiles(32, 64) <= 256) return Q8Form::Narrow;
    if (tiles(64, 64) <= 256) return Q8Form::Square;
    if (tiles(32, 128) <= 256) return Q8Form::Rows32;
    if (grid(64, 64) <= 512) return Q8Form::Square;
    return Q8Form::Small3;
}

}  // namespace s2x
