"""Products of many rows whose last or only round of workgroups takes tiles of 192 or 224 activation rows (q8_gemm_wide.hip), against
the f64 product over the exactly dequantised weights: one row past a tile, a row short of one, odd N, two rounds, behind tiles of 256 rows,
all output forms."""
import ctypes as C

import pytest

torch = pytest.importorskip("torch")

from luminal_amd import capi, synth  # noqa: E402
from luminal_amd.quantized import Q8Weight, QuantizedMatmul, QuantizedMatmulBf16  # noqa: E402

DEV = "cuda:0"
# By the height of the last or only round's tiles: 7 x 24 + 1 row, 4 tiles + 1 row of 40, 10 x 24, two rounds of 56, and behind 32 and 31
# column tiles of 256 rows; 9 tiles - 1 row, 9 tiles + 1 row
SIZES = {192: [(1345, 6141, 320), (769, 9999, 576), (1793, 6144, 256), (1700, 14336, 320), (1979, 12800, 320), (1757, 14079, 320)],
         224: [(2015, 6140, 320), (2017, 6140, 448)]}
ALL = [s for sizes in SIZES.values() for s in sizes]


def test_sizes_take_tiles_of_their_height():
    lib, out = capi.load_library(), (C.c_int32 * 3)()
    for height, sizes in SIZES.items():
        for s in sizes:
            capi.check(lib.lhip_q8_0_matmul_plan(*s, 2, (1 << 64) - 1, out), "plan")
            assert tuple(out) == (3, height, 1), s


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", ALL)
def test_against_f64(m, n, k):
    lib, st = capi.load_library(), torch.cuda.current_stream().cuda_stream
    w = Q8Weight.from_raw(synth.q8_0_raw_blocks(*synth.q8_0_random(n, k, seed=m)), n, k, DEV)
    gen = torch.Generator(device=DEV).manual_seed(n)
    x = torch.randn((m, k), device=DEV, generator=gen).to(torch.bfloat16)
    wd = w.dequantize().double()
    want, bound = x.double() @ wd.t(), (x.double().abs() @ wd.abs().t()) * (k // 32 + 33) * 2.0 ** -24  # f32 additions
    y = torch.full((m, n), float("nan"), device=DEV)
    capi.check(lib.lhip_q8_0_matmul_bf16_f32out(w.planar.data_ptr(), x.data_ptr(), y.data_ptr(), m, n, k, st), "f32out")
    assert bool(((y.double() - want).abs() <= bound).all())
    assert torch.equal(QuantizedMatmulBf16().process(x, w).view(torch.int16), y.to(torch.bfloat16).view(torch.int16))
    if n % 4 == 0:
        act, of_y = (torch.full((m, n // 2), float("nan"), device=DEV, dtype=torch.bfloat16) for _ in range(2))
        capi.check(lib.lhip_q8_0_matmul_bf16_swiglu(w.planar.data_ptr(), x.data_ptr(), act.data_ptr(), m, n, k, st), "swiglu")
        capi.check(lib.lhip_swiglu_f32_bf16out(y.data_ptr(), of_y.data_ptr(), m, n // 2, 1, st), "swiglu of f32")
        assert torch.equal(act.view(torch.int16), of_y.view(torch.int16))
    x16 = x.to(torch.float16)
    y16, want = QuantizedMatmul().process(x16, w).double(), x16.double() @ wd.t()
    assert bool(((y16 - want).abs() <= bound * 1.01 + want.abs() * 2.0 ** -11 + 2.0 ** -25).all())
