"""Shapes that take each tile form of the GEMMs, for the CPU test of the rules
and the GPU tests of the forms."""
# the int8 GEMM's latency forms: (form, M, N, plain epilogue)
LATENCY_SHAPES = [
    ("Lone", 31, 65, True), ("Lone", 33, 1152, True),
    ("Narrow", 300, 1003, True), ("Narrow", 321, 1001, True),
    ("Square", 700, 1003, True), ("Square", 1400, 500, True),
    ("Rows32", 200, 4300, True), ("Rows32", 150, 6403, True),
    ("Small3", 1801, 1153, True), ("Small3", 1801, 1153, False),
    ("Small4", 33, 65, False), ("Small4", 700, 1003, False),
]

# the F16 GEMM's: (form, M, K, N), 8 stages of 64 halves and more
F16_SHAPES = [
    ("Small", 130, 600, 129), ("Small", 64, 4304, 1152),
    ("Mid", 16449, 600, 100), ("Mid", 16449, 1001, 100), ("Mid", 2916, 4304, 1152),
    ("Wide", 32897, 600, 100),
]
# rows of the so400m tower's fc2 (N = 1,152) that take them: 1, 4 and 32
# images of 729 patches
F16_TOWER_ROWS = {"Small": 729, "Mid": 4 * 729, "Wide": 32 * 729}
