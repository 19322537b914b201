"""Products whose workgroups walk all of K (q8_gemm_deep.hip), by the plain operators at sizes that take that kernel, against the f64
product over the exactly dequantised weights: every tile of it, ragged rows and columns, odd N, K of whole quads of blocks and with a pair
left over, of fewer quads than a workgroup walks side by side, and all output forms."""
import ctypes as C

import pytest
import torch

from luminal_amd import capi, synth
from luminal_amd.quantized import Q8Weight, QuantizedMatmul, QuantizedMatmulBf16

DEV = "cuda:0"
# By tile (activation rows x weight rows): 32, 48, 64, 96 and 128 x 32, then x 64
BOTH = [(49, 3725, 512), (130, 2068, 512), (255, 1696, 576), (161, 2750, 576), (193, 2568, 512),
        (129, 2480, 512), (130, 3660, 576), (257, 2728, 512), (130, 5452, 512), (97, 8339, 576)]
BF16_ONLY = [(300, 36, 448), (17, 1001, 576), (130, 257, 320), (200, 1030, 1152), (132, 2880, 2880),
             (76, 3224, 768), (101, 468, 576), (112, 1196, 704)]


def kernel_of(m, n, k, activations):
    lib, out = capi.load_library(), (C.c_int32 * 3)()
    capi.check(lib.lhip_q8_0_matmul_plan(m, n, k, activations, (1 << 64) - 1, out), "lhip_q8_0_matmul_plan")
    return out[0], out[2]


def test_sizes_reach_the_kernel():
    assert all(kernel_of(*s, 2) == (4, 1) for s in BOTH + BF16_ONLY)
    assert all(kernel_of(*s, 1) == (4, 1) for s in BOTH)


def operands(m, n, k, dtype):
    w = Q8Weight.from_raw(synth.q8_0_raw_blocks(*synth.q8_0_random(n, k, seed=m + n)), n, k, DEV)
    x = torch.randn((m, k), device=DEV, generator=torch.Generator(device=DEV).manual_seed(k)).to(dtype)
    xd, wd = x.double(), w.dequantize().double()
    # f32 additions: 32 of a block, then the blocks (four chains and their sum), each of 2^-24 of what has been added so far
    return w, x, xd @ wd.t(), (xd.abs() @ wd.abs().t()) * (k // 32 + 36) * 2.0 ** -24


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", BOTH + BF16_ONLY)
def test_bf16_forms(m, n, k):
    w, x, want, bound = operands(m, n, k, torch.bfloat16)
    lib, st = capi.load_library(), torch.cuda.current_stream().cuda_stream
    y = torch.full((m, n), float("nan"), device=DEV)
    capi.check(lib.lhip_q8_0_matmul_bf16_f32out(w.planar.data_ptr(), x.data_ptr(), y.data_ptr(), m, n, k, st), "f32out")
    assert bool(((y.double() - want).abs() <= bound).all())
    y16 = QuantizedMatmulBf16().process(x, w)
    assert torch.equal(y16.view(torch.int16), y.to(torch.bfloat16).view(torch.int16))
    if n % 4 == 0:
        act, of_y = (torch.full((m, n // 2), float("nan"), device=DEV, dtype=torch.bfloat16) for _ in range(2))
        capi.check(lib.lhip_q8_0_matmul_bf16_swiglu(w.planar.data_ptr(), x.data_ptr(), act.data_ptr(), m, n, k, st), "swiglu")
        capi.check(lib.lhip_swiglu_f32_bf16out(y.data_ptr(), of_y.data_ptr(), m, n // 2, 1, st), "swiglu of f32")
        assert torch.equal(act.view(torch.int16), of_y.view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", BOTH)
def test_f16(m, n, k):
    w, x, want, bound = operands(m, n, k, torch.float16)
    y = QuantizedMatmul().process(x, w)
    assert bool(((y.double() - want).abs() <= bound + want.abs() * 2.0 ** -11 + 2.0 ** -25).all())


@pytest.mark.gpu
def test_an_infinity_and_a_nan_stay_in_their_rows():
    """Steps behind the end of K read the last pair of blocks again and must not multiply it."""
    m, n, k = 130, 257, 320
    w, x, want, bound = operands(m, n, k, torch.bfloat16)
    x[3, k - 1], x[70, 0] = float("inf"), float("nan")
    y = QuantizedMatmulBf16().process(x, w).double()
    rest = [r for r in range(m) if r not in (3, 70)]
    assert bool(((y - want).abs() <= bound + want.abs() * 2.0 ** -8)[rest].all())
    assert bool(y[70].isnan().all()) and not bool(y[3].isfinite().any())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(10, 2880, 2880), (8, 6000, 1600), (23, 4831, 1024)])
def test_f16_of_a_few_rows(m, n, k):
    """Fewer rows than a tile, that would be matvecs otherwise; the plain C call, which has no workspace, gives the operator's bits."""
    assert kernel_of(m, n, k, 1) == (4, 1)
    w, x, want, bound = operands(m, n, k, torch.float16)
    y = QuantizedMatmul().process(x, w)
    assert bool(((y.double() - want).abs() <= bound + want.abs() * 2.0 ** -11 + 2.0 ** -25).all())
    plain = torch.full_like(y, float("nan"))
    capi.check(capi.load_library().lhip_q8_0_matmul_f16(w.planar.data_ptr(), x.data_ptr(), plain.data_ptr(), m, n, k,
                                                        torch.cuda.current_stream().cuda_stream), "f16")
    assert torch.equal(plain.view(torch.int16), y.view(torch.int16))
