"""The tile kernel for many activation rows (lhip_q8_0_matmul_bf16_cfg tile 0): the sizes where its pipeline, its mixed
tiles and its stores have an edge, against the f64 product of the oracle.

A result is a sum of K exact products with f32 additions, at most K / 32 + 33 of them in a chain: relative to the sum of
the terms' magnitudes the error is below (K / 32 + 33) * 2^-24, which the f32 output is held to element by element; the
bf16 output is that rounded once.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from luminal_amd import capi, synth  # noqa: E402
from luminal_amd.quantized import Q8Weight, QuantizedMatmulBf16  # noqa: E402

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def problem(oracle, m, n, k):
    qs, d = synth.q8_0_random(n, k, seed=m + n + k)
    bits = oracle.f32_to_bf16_bits(synth.activations(m, k, seed=m * n))
    wf = oracle.q8_0_dequant(synth.q8_0_raw_blocks(qs, d), qs.size).reshape(qs.shape)
    w = Q8Weight.from_raw(synth.q8_0_raw_blocks(qs, d), n, k, DEV)
    x = torch.from_numpy(bits.view(np.int16)).to(DEV).view(torch.bfloat16)
    xf = oracle.bf16_bits_to_f32(bits)
    bound = oracle.matmul_f64(np.abs(xf), np.abs(wf)) * (k // 32 + 33) * 2.0 ** -24
    return w, x, oracle.matmul_f64(xf, wf), bound


# K of 1, 2, 3 and 5 tiles (fewer and more than the stages of the pipeline); one row, one row less and more than a tile;
# N below a wave's 32 rows, one less and more than a tile, odd (two-byte stores) and even (words); last: tiles of both
# heights in one launch, both ragged
@pytest.mark.parametrize("m,n,k", [(1, 1, 64), (127, 31, 128), (129, 255, 192), (257, 257, 320), (300, 258, 64),
                                   (128, 512, 1024), (1100, 8198, 128)])
def test_large_tiles_at_their_edges(oracle, m, n, k):
    w, x, truth, bound = problem(oracle, m, n, k)
    y16 = QuantizedMatmulBf16(0).process(x, w).float().cpu().numpy().astype(np.float64)
    assert np.all(np.abs(y16 - truth) <= bound + np.abs(truth) * 2.0 ** -8)


def test_output_forms_agree_and_uneven_slices_hold(oracle):
    """1100 x 8196 x 128 takes the large tiles for every output form: bf16 is the f32 result rounded once and SwiGLU is
    lhip_swiglu_f32_bf16out of it.  600 x 1000 x 832 is cut into uneven slices of K."""
    lib = capi.load_library()
    s = torch.cuda.current_stream().cuda_stream
    for m, n, k in ((1100, 8196, 128), (600, 1000, 832)):
        w, x, truth, bound = problem(oracle, m, n, k)
        y32 = torch.full((m, n), float("nan"), device=DEV)
        y16 = torch.empty((m, n), device=DEV, dtype=torch.bfloat16)
        act, want = (torch.empty((m, n // 2), device=DEV, dtype=torch.bfloat16) for _ in range(2))
        capi.check(lib.lhip_q8_0_matmul_bf16_f32out(w.planar.data_ptr(), x.data_ptr(), y32.data_ptr(), m, n, k, s), "f32")
        capi.check(lib.lhip_q8_0_matmul_bf16(w.planar.data_ptr(), x.data_ptr(), y16.data_ptr(), m, n, k, s), "bf16")
        capi.check(lib.lhip_q8_0_matmul_bf16_swiglu(w.planar.data_ptr(), x.data_ptr(), act.data_ptr(), m, n, k, s), "swiglu")
        capi.check(lib.lhip_swiglu_f32_bf16out(y32.data_ptr(), want.data_ptr(), m, n // 2, 1, s), "swiglu of f32")
        torch.cuda.synchronize()
        assert np.all(np.abs(y32.cpu().numpy().astype(np.float64) - truth) <= bound)
        assert torch.equal(y32.to(torch.bfloat16).view(torch.int16), y16.view(torch.int16))
        assert torch.equal(act.view(torch.int16), want.view(torch.int16))
