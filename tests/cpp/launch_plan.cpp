// The launch rules of csrc/s2x_plan.h, for tests/test_launch_plan.py.
#include "s2x_plan.h"

extern "C" {
void plan_f16_operand_grid(int64_t rows, int64_t ld, int64_t *out) {
    const s2x::F16OperandGrid g = s2x::f16_operand_grid(rows, ld);
    out[0] = g.lg_lanes, out[1] = g.col_blocks, out[2] = g.blocks;
}
int plan_f16_w_in_place(uintptr_t w, uintptr_t y, uintptr_t ws, int64_t K, int64_t N, int64_t M) {
    return s2x::f16_w_in_place(w, y, ws, K, N, M);
}
void plan_f16_mul_mat(int64_t K, int64_t N, int64_t M, int w_in_place, int64_t *out) {
    const s2x::F16MulMatPlan p = s2x::f16_mul_mat_plan(K, N, M, w_in_place != 0);
    out[0] = p.w_direct, out[1] = p.ldx16, out[2] = p.ldw, out[3] = p.x_off, out[4] = p.total;
}
int plan_f16_ld_ok(int64_t ld) { return s2x::f16_ld_ok(ld); }
int plan_q8_form(int64_t M, int64_t N, int plain, int64_t n_split) {
    return (int)s2x::q8_form(M, N, plain != 0, n_split);
}
int plan_f16_form(int64_t M, int64_t N, int64_t ldx) { return (int)s2x::f16_form(M, N, ldx); }
}
