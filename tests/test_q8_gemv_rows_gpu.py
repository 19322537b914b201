"""Matvecs of several activation rows a pass (q8_gemv_rows.hip), by the plain operators at sizes that take them: every row's result is bit
for bit that of the one-shot matvec kernel, which is held against the f64 product elsewhere; an f16 result is that of the widened
activations rounded once."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from luminal_amd import capi, synth  # noqa: E402
from luminal_amd.quantized import Q8Weight, QuantizedMatmul  # noqa: E402

DEV = "cuda:0"
ONE_SHOT = QuantizedMatmul(1, 1, 0, 4)

# Every number of rows a pass and passes left short; one and two slices a step, steps past K; row groups fewer than waves, one past a round of
# workgroups; the activations of one row filling a pass; K of one slice
SIZES = [(2, 3073, 4096), (3, 4096, 4096), (4, 2051, 4096), (5, 1501, 2048), (5, 2880, 2880), (1, 7, 10272), (5, 259, 5152), (1, 1001, 14304),
         (24, 260, 3136), (13, 300, 8000), (2, 4096, 14336), (3, 1601, 13312), (1, 33, 20512), (2, 1065, 40928), (12, 1100, 2016),
         (11, 1601, 1024), (3, 4097, 3072), (2, 12001, 1504), (7, 2050, 5120), (2, 848, 16384), (2, 360, 40960)]
F32_ONLY = [(11, 2001, 992), (11, 1100, 1056), (2, 8193, 1056)]


def rows_of_pass(m, n, k, activations):
    """Activation rows that a pass of the matvecs takes by the library's answer; 0: another kernel, or a matvec a row."""
    lib, out = capi.load_library(), (C.c_int32 * 3)()
    capi.check(lib.lhip_q8_0_matmul_plan(m, n, k, activations, lib.lhip_q8_0_matmul_workspace_nbytes(m, n, k), out), "plan")
    return out[1] if out[0] == 0 else 0


def test_sizes_reach_the_kernel():
    for activations, sizes in ((0, SIZES + F32_ONLY), (1, SIZES)):
        rows = [rows_of_pass(*s, activations) for s in sizes]
        assert all(rows), [s for s, r in zip(sizes, rows) if r == 0]
        assert set(rows) == {1, 2, 3, 4, 5}
    assert rows_of_pass(1, 4096, 4096, 0) == 0 and rows_of_pass(64, 4096, 4096, 0) == 0


def same(a, b):
    return bool(((a == b) | (a.isnan() & b.isnan())).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", SIZES + F32_ONLY)
def test_rows_of_a_pass_have_the_one_row_bits(m, n, k):
    qs, d = synth.q8_0_random(n, k, seed=m + n + k)
    w = Q8Weight.from_raw(synth.q8_0_raw_blocks(qs, d), n, k, DEV)
    x = torch.from_numpy(synth.activations(m, k, seed=m * n)).to(DEV)
    assert torch.equal(QuantizedMatmul().process(x, w), ONE_SHOT.process(x, w))
    # (halves that are aligned to 8 bytes only)
    x16 = torch.empty(m * k + 4, dtype=torch.float16, device=DEV)[4:].view(m, k).copy_(x)
    assert torch.equal(QuantizedMatmul().process(x16, w), ONE_SHOT.process(x16.float(), w).half())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(3, 2880, 2880), (2, 77, 4128), (2, 4096, 4096)])
def test_values_that_are_not_finite_stay_in_their_row(m, n, k):
    """Infinities and NaN among the activations and the scales, the last block's among them: lanes that lie behind a ragged K add nothing."""
    qs, d = synth.q8_0_random(n, k, seed=5)
    qs[:, 3] = np.arange(n) % 3 - 1
    d[1, 0], d[2, -1], d[3, 0] = np.inf, np.inf, np.nan
    w = Q8Weight.from_raw(synth.q8_0_raw_blocks(qs, d), n, k, DEV)
    x = torch.from_numpy(synth.activations(m, k, seed=6)).to(DEV)
    x[1, 3], x[0, k - 1] = float("inf"), 65504.0
    y = QuantizedMatmul().process(x, w)
    assert same(y, ONE_SHOT.process(x, w)) and bool(y[0, 0].isfinite()) and bool(y[0, 3].isnan())
    assert not y[:, 1:4].isfinite().any()  # (an infinite scale meets the block's halves, whose sums may differ in sign: infinite or NaN)
    y16 = QuantizedMatmul().process(x.half(), w)
    assert same(y16, ONE_SHOT.process(x.half().float(), w).half())
