// The launch rules of csrc/s2x_plan.h, for tests/test_launch_plan.py.
#include "s2x_plan.h"

extern "C" {
void plan_f16_operand_grid(int64_t rows, int64_t ld, int64_t *out) {
    const s2x::F16OperandGrid g = s2x::f16_operand_grid(rows, ld);
    out[0] = g.lg_lanes, out[1] = g.col_blocks, out[2] = g.blocks;
}
}
