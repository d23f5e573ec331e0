"""The rules by which the launchers choose grids and layouts from sizes
(csrc/s2x_plan.h), compiled for the CPU."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from gemm_forms import F16_SHAPES, F16_TOWER_ROWS, LATENCY_SHAPES

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "hbd-siglip2.cpp_amd", "csrc")

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    so = tmp_path_factory.mktemp("plan") / "launch_plan.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, "-o", str(so),
                    os.path.join(HERE, "cpp", "launch_plan.cpp")], check=True)
    return ctypes.CDLL(str(so))


def _operand_grid(plan, rows, ld):
    out = (ctypes.c_int64 * 3)()
    plan.plan_f16_operand_grid(ctypes.c_int64(rows), ctypes.c_int64(ld), out)
    return tuple(out)  # log2 of the lanes per row, blocks along a row, blocks


def _up(a, b):
    return (a + b - 1) // b * b


@pytest.mark.parametrize("rows", [1, 3, 4, 63, 64, 65, 257])
@pytest.mark.parametrize("ld", [8, 16, 24, 32, 64, 72, 256, 264, 512, 520, 544, 1024, 4352])
def test_f16_operand_grid_covers_each_chunk_once(plan, rows, ld):
    lg, ncb, blocks = _operand_grid(plan, rows, ld)
    bid, tid = np.divmod(np.arange(blocks * 256), 256)
    row = bid // ncb * (256 >> lg) + (tid >> lg)
    c = (bid % ncb) * (8 << lg) + (tid & ((1 << lg) - 1)) * 8
    ok = (row < rows) & (c < ld)
    assert np.array_equal(np.unique(row[ok] * ld + c[ok]), np.arange(0, rows * ld, 8))
    assert ok.sum() == rows * ld // 8


def test_f16_operand_grid_takes_rows_up_to_the_launch_limit(plan):
    # HIP refuses 2^32 threads along x.  A thread per 4 halves of rows padded
    # to 32 stays below that up to 2^34 / K_pad rows; the grid must take all
    # of those, at the stride of whole 128-byte lines too (2^26 rows of K = 8
    # among them, where 64 lanes a row are 2^32 threads)
    for K in (*range(8, 2200, 8), 4304, 65536, 1 << 20):
        k_pad = _up(K, 32)
        rows = min(1 << 30, ((1 << 32) - 256) * 4 // k_pad)
        for ld in (k_pad, _up(K, 64)):
            assert _operand_grid(plan, rows, ld)[2] * 256 < 1 << 32, (K, ld, rows)


def _w_in_place(plan, w, y, K, N, M, ws=1 << 51):
    return bool(plan.plan_f16_w_in_place(*(ctypes.c_uint64(v) for v in (w, y, ws)),
                                         *(ctypes.c_int64(v) for v in (K, N, M))))


def _f16_plan(plan, K, N, M, w_align16):
    out = (ctypes.c_int64 * 5)()
    in_place = w_align16 and _w_in_place(plan, 1 << 20, 1 << 50, K, N, M)
    plan.plan_f16_mul_mat(*(ctypes.c_int64(v) for v in (K, N, M)), int(in_place), out)
    return tuple(out)


def test_f16_weight_is_read_in_place_only_beside_y(plan):
    K, N, M, w = 64, 10, 7, 1 << 20
    end, size = w + N * K * 2, M * N * 4
    assert _w_in_place(plan, w, end, K, N, M) and _w_in_place(plan, w, w - size, K, N, M)
    # y over the weight, from its first byte to its last: the rows are copied
    # first, as the result overwrites them
    for y in (w, w + 4, end - 4, w - size + 4, w - 4):
        assert not _w_in_place(plan, w, y, K, N, M), y - w
    # the same for the workspace, where X's rows are written first (a weight
    # with K % 32 == 0 may lie where its own copy goes, at the front of it)
    far, total = 1 << 50, _f16_plan(plan, K, N, M, False)[4]
    assert _w_in_place(plan, w, far, K, N, M, end) and _w_in_place(plan, w, far, K, N, M, w - total)
    for ws in (w, w + 256, w - 256, w - total + 256):
        assert not _w_in_place(plan, w, far, K, N, M, ws), ws - w
    assert not _w_in_place(plan, w + 8, end + 8, K, N, M)   # alignment
    assert not _w_in_place(plan, w, end + 4096, 63, N, M)   # of every row


def test_f16_mul_mat_layouts_fit_the_workspace_and_the_gemm(plan):
    # (K = 8,388,552 among them: its rows padded to 32 are within the GEMM's
    # stride limit, rows of whole lines are not)
    for K in (1, 7, 8, 24, 32, 40, 64, 72, 1001, 1076, 1152, 4304, 8388480, 8388488, 8388544, 8388552, 8388576):
        k_pad = _up(K, 32)
        assert plan.plan_f16_ld_ok(ctypes.c_int64(k_pad))
        for N, M in ((1, 1), (1, 3), (2, 300), (300, 2), (1152, 729)):
            for al in (0, 1):
                direct, ldx, ldw, x_off, total = _f16_plan(plan, K, N, M, al)
                assert total == _up(N * k_pad * 2, 256) + _up(M * k_pad * 2, 256)  # part of the interface
                assert direct == (al and K % 8 == 0)
                assert ldw == (K if direct else k_pad) and ldx >= K and ldx % 8 == 0
                assert plan.plan_f16_ld_ok(ctypes.c_int64(ldx)), (K, N, M, al)
                assert x_off % 256 == 0 and x_off + M * ldx * 2 <= total
                assert direct or x_off >= N * ldw * 2  # the repacked rows lie in front
    assert _f16_plan(plan, 4304, 1152, 2916, 1)[1] == 4352  # whole lines
    assert not plan.plan_f16_ld_ok(ctypes.c_int64(8388608))


Q8_FORMS = ["Wide", "Lone", "Narrow", "Square", "Rows32", "Small4", "Small3"]


def _q8_form(plan, M, N, plain=True, n_split=1):
    return Q8_FORMS[plan.plan_q8_form(ctypes.c_int64(M), ctypes.c_int64(N), int(plain), ctypes.c_int64(n_split))]


@pytest.mark.parametrize("form,M,N,plain", LATENCY_SHAPES)
def test_latency_shapes_take_their_form(plan, form, M, N, plain):
    # the shapes of the GPU tests of each tile form
    assert _q8_form(plan, M, N, plain) == form


@pytest.mark.parametrize("n_split", [1, 2, 4, 16])
def test_q8_form_fills_the_cus_once(plan, n_split):
    # a plain product within one workgroup per CU of some form is not given
    # to one that puts two on a few CUs (M = 200, N = 4,304 took 23.8 us that
    # way, 18.2 in 32 x 128 tiles); a K split has n_split workgroups per tile
    dims = {"Lone": (32, 32), "Narrow": (32, 64), "Square": (64, 64), "Rows32": (32, 128)}
    for M in range(9, 1500, 13):
        for N in (64, 256, 768, 1152, 2304, 3456, 4304):
            tiles = {f: -(-M // bm) * -(-N // bn) * n_split for f, (bm, bn) in dims.items()}
            got = _q8_form(plan, M, N, True, n_split)
            if min(tiles.values()) <= 256:
                assert tiles[got] <= 256, (M, N, got, tiles)
            assert _q8_form(plan, M, N, False) in ("Wide", "Small4", "Small3")


def test_f16_shapes_take_their_form(plan):
    shapes = [(f, M, K, N) for f, M, K, N in F16_SHAPES]
    shapes += [(f, M, 4304, 1152) for f, M in F16_TOWER_ROWS.items()]
    for form, M, K, N in shapes:
        got = plan.plan_f16_form(ctypes.c_int64(M), ctypes.c_int64(N), ctypes.c_int64(_up(K, 64)))
        assert ["Small", "Mid", "Wide"][got] == form, (M, K, N)
