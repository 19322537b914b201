"""Whether the sizes of the matmul tests reach the kernels, and the strips, tiles and K slices, that they are listed for.  No GPU."""
import ctypes as C

import pytest

from luminal_amd import capi
from matmul_shapes import ROWS, STREAMED_BF16, STREAMED_BF16_ANY_K, STREAMED_F32_F16

TYPES = {"f32": 0, "f16": 1, "bf16": 2}
PLAIN = (1 << 64) - 1
MATVEC, STREAM, ROWS_KERNEL, TILES = 0, 1, 2, 3


def plan(m, n, k, dtype, workspace=False):
    """(kernel, weight rows of a workgroup, K slices), of the plain call or with the recommended workspace."""
    lib, out = capi.load_library(), (C.c_int32 * 3)()
    room = PLAIN
    if workspace:
        room = lib.lhip_q8_0_matmul_bf16_workspace_nbytes(m, n, k, 0) if dtype == "bf16" else lib.lhip_q8_0_matmul_workspace_nbytes(m, n, k)
    capi.check(lib.lhip_q8_0_matmul_plan(m, n, k, TYPES[dtype], room, out), "lhip_q8_0_matmul_plan")
    return tuple(out)


def cuts(plans):
    """The (weight rows, whether K is sliced) that occur."""
    return {(rows, slices > 1) for _, rows, slices in plans}


def test_strips_of_the_weight_streaming_kernel():
    plans = [plan(*s, "bf16") for s in STREAMED_BF16]
    assert {p[0] for p in plans} == {STREAM}
    assert cuts(plans) == {(rows, sliced) for rows in (32, 48, 64, 112, 128) for sliced in (False, True)}
    for dtype in ("f32", "f16"):
        plans = [plan(*s, dtype) for s in STREAMED_F32_F16]
        assert {p[0] for p in plans} == {STREAM}, list(zip(STREAMED_F32_F16, plans))
        assert cuts(plans) == {(rows, sliced) for rows in (32, 48, 64, 128) for sliced in (False, True)}


def test_strips_of_the_weight_streaming_kernel_for_any_k():
    plans = [(plan(*s, "bf16"), plan(*s, "bf16", workspace=True)) for s in STREAMED_BF16_ANY_K]
    assert all(plain[0] == STREAM for plain, _ in plans) and sum(ws[0] == STREAM for _, ws in plans) >= len(plans) - 1
    assert all(plain[2] == 1 for plain, _ in plans)  # nothing is kept outside the outputs
    assert cuts(p for both in plans for p in both if p[0] == STREAM) == {(rows, sliced) for rows in (32, 64, 128) for sliced in (False, True)}


@pytest.mark.parametrize("dtype", ["f32", "f16"])
def test_tiles_of_the_kernel_for_several_rows(dtype):
    plans = [plan(*s, dtype, workspace=True) for s in ROWS[dtype]]
    assert {p[0] for p in plans} == {ROWS_KERNEL}, list(zip(ROWS[dtype], plans))
    assert cuts(plans) == {(rows, sliced) for rows in (128, 192, 224, 256) for sliced in (False, True)}, list(zip(ROWS[dtype], plans))


def test_f16_products_of_a_large_ragged_matrix_stay_with_k_slices():
    """Weights that no cache holds: the kernel that walks all of K was up to a fifth behind there, ahead for smaller ones."""
    for s in ((6, 8369, 6144), (11, 5048, 11904), (32, 5204, 13888), (10, 12398, 10880)):
        assert plan(*s, "f16", workspace=True)[0] == ROWS_KERNEL, s
    for s in ((45, 2880, 2880), (23, 4830, 1024), (251, 848, 5184), (9, 3208, 2304)):
        assert plan(*s, "f16", workspace=True)[0] == 4, s


def test_matvecs_of_several_rows_a_pass_where_they_pay():
    """Whole slices of a K beyond 12288, where a matvec a row was up to twice as slow; a short K by the further rows."""
    for s, t in (((2, 360, 40960), "f16"), ((3, 512, 40960), "f32"), ((2, 848, 16384), "f32"), ((4, 280, 14336), "f16"), ((2, 804, 12288), "f16"),
                 ((4, 2862, 1024), "f32"), ((4, 8020, 512), "f32")):
        assert plan(*s, t)[0] == MATVEC and plan(*s, t)[1] > 0, (s, t)
    for s in ((3, 167, 12288), (2, 240, 4096), (3, 5195, 416)):
        assert plan(*s, "f32") == (MATVEC, 0, 1), s


def test_the_matvec_of_one_row_of_a_ragged_k():
    """The kernel of several rows also takes one where its waves have at most one weight row each (up to a seventh sooner), not for twice as many."""
    for n, k, t, rows in ((160, 3552, "f32", 1), (1920, 3936, "f32", 1), (1141, 4608, "f16", 1), (2380, 5088, "f32", 0), (3576, 4704, "f16", 0), (4000, 4608, "f32", 1), (7084, 3840, "f16", 0), (8316, 3904, "f16", 1),
                          (1920, 3040, "f32", 0), (1141, 4064, "f16", 0)):
        assert plan(1, n, k, t) == (MATVEC, rows, 1), (n, k, t)


def test_a_single_row_is_a_matvec_for_any_size():
    """Also where K is short and the weight rows are very many (128256 x 288 went to the matrix cores)."""
    lib = capi.load_library()
    for n in (1, 1000, 14336, 65536, 128256, 262144):
        for k in (256, 288, 512, 1056, 2880, 8000, 14368, 40992, 70016):
            assert lib.lhip_q8_0_matmul_workspace_nbytes(1, n, k) == 0, (n, k)
            for dtype in ("f32", "f16"):
                assert plan(1, n, k, dtype)[0] == plan(1, n, k, dtype, workspace=True)[0] == MATVEC, (n, k, dtype)


def test_ragged_products_of_a_very_long_k():
    """Where matvecs take several passes over the weights, or LDS holds no row of their activations, K slices end up to 2.6 times sooner."""
    for s, t in (((3, 5796, 56672), "f32"), ((3, 1688, 52544), "f16"), ((3, 11448, 33696), "f16"), ((3, 18824, 14976), "f32")):
        assert plan(*s, t, workspace=True)[0] == ROWS_KERNEL, (s, t)
    for s, t in (((11, 1928, 3648), "f32"), ((3, 6808, 22592), "f16"), ((2, 16514, 34464), "f32"), ((3, 95540, 544), "f32"),
                 ((3, 29325, 7680), "f16")):
        assert plan(*s, t, workspace=True)[0] == MATVEC, (s, t)
    for s in ((8, 27324, 10368), (6, 16272, 30336)):  # (weights beyond any cache: what they cost from memory is in the estimates of both)
        assert plan(*s, "f16", workspace=True)[0] == 4, s


def test_no_room_is_asked_for_where_neither_type_keeps_anything_in_it():
    """A K outside the weight-streaming kernel's shapes: the recommended workspace is used by the f32 or the f16 call, or it is 0."""
    lib, asked = capi.load_library(), 0
    for m in (2, 5, 6, 8, 10, 12, 24, 45, 128):
        for n in (256, 1000, 2880, 6001, 10944, 14336):
            for k in (544, 576, 960, 1600, 2880, 4160, 8000):
                if lib.lhip_q8_0_matmul_workspace_nbytes(m, n, k):
                    asked += 1
                    assert any(plan(m, n, k, t, workspace=True)[2] != 1 for t in ("f32", "f16")), (m, n, k)
    assert asked > 50


def test_plan_errors():
    lib, out = capi.load_library(), (C.c_int32 * 3)()
    assert lib.lhip_q8_0_matmul_plan(1, 32, 32, 0, PLAIN, None) == capi.LHIP_ERR_NULL_PTR
    for bad in ((0, 32, 32, 0), (1, 0, 32, 0), (1, 32, 33, 0), (1, 32, 32, 3), (1, 32, 32, -1)):
        assert lib.lhip_q8_0_matmul_plan(*bad, PLAIN, out) == capi.LHIP_ERR_INVALID_SHAPE
    assert lib.lhip_q8_0_matmul_plan(1, 32, 32, 2, PLAIN, out) == capi.LHIP_ERR_UNSUPPORTED  # bf16: K in steps of 64
    assert plan(1, 4096, 4096, "f32") == (MATVEC, 0, 1) and plan(2048, 14336, 4096, "bf16")[0] == TILES
