"""The int8 GEMM's tile forms and shapes that take them (form, M, N, plain
epilogue), for the CPU test of the rule and the GPU tests of the forms."""
LATENCY_SHAPES = [
    ("Lone", 31, 65, True), ("Lone", 33, 1152, True),
    ("Narrow", 300, 1003, True), ("Narrow", 321, 1001, True),
    ("Square", 700, 1003, True), ("Square", 1400, 500, True),
    ("Rows32", 200, 4300, True), ("Rows32", 150, 6403, True),
    ("Small3", 1801, 1153, True), ("Small3", 1801, 1153, False),
    ("Small4", 33, 65, False), ("Small4", 700, 1003, False),
]
