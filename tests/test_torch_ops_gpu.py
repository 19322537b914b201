"""The operators' native host path (host/torch_ops.cpp) against the Python one: the same bits, the same errors, and what it leaves
to the other."""
import pytest

torch = pytest.importorskip("torch")

from luminal_amd import capi, quantized, synth  # noqa: E402
from luminal_amd.quantized import Q8Weight, QuantizedMatmul, QuantizedMatmulBf16  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def weight(n, k):
    return Q8Weight.from_raw(synth.q8_0_raw_blocks(*synth.q8_0_random(n, k, seed=n + k)), n, k, DEV)


def through_python(monkeypatch, op, x, w):
    with monkeypatch.context() as m:
        m.setattr(quantized, "_native_matmul", lambda *_: None)
        return op.process(x, w)


def native_ops():
    """The extension; its tests are skipped where it is not built (the operators then run through ctypes)."""
    return pytest.importorskip("luminal_amd._torch_ops")


def test_the_native_path_runs_where_it_is_built():
    assert quantized._native_matmul is native_ops().quantized_matmul


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("shape,n,k", [((1, 512), 256, 512), ((3, 1024), 260, 1024), ((2, 3, 5, 704), 129, 704), ((45, 2880), 2880, 2880),
                                       ((130, 1024), 516, 1024), ((64,), 8, 64)])
def test_same_bits_as_the_python_path(monkeypatch, dtype, shape, n, k):
    op, w = (QuantizedMatmulBf16() if dtype == torch.bfloat16 else QuantizedMatmul()), weight(n, k)
    x = torch.randn(shape, device=DEV).to(dtype)
    device = torch.cuda.current_device()
    native = native_ops().quantized_matmul(x, w.planar, n, k, dtype == torch.bfloat16, device, torch.cuda.current_stream().cuda_stream)
    assert native is not None and native.shape == (*shape[:-1], n) and native.dtype == dtype
    want = through_python(monkeypatch, op, x, w)
    assert torch.equal(native.view(torch.uint8), want.view(torch.uint8))
    # strided activations, and a stream of one's own
    wide = torch.zeros((*shape[:-1], 2 * k), dtype=dtype, device=DEV)
    wide[..., ::2] = x
    assert torch.equal(op.process(wide[..., ::2], w).view(torch.uint8), want.view(torch.uint8))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = op.process(x, w)
    side.synchronize()
    assert torch.equal(y.view(torch.uint8), want.view(torch.uint8))


@pytest.mark.parametrize("op,good", [(QuantizedMatmul(), torch.float32), (QuantizedMatmulBf16(), torch.bfloat16)])
def test_what_is_refused_stays_refused(op, good):
    w = weight(64, 128)
    for bad in (torch.float32, torch.float16, torch.bfloat16, torch.float64, torch.int8):
        if bad != good and not (good == torch.float32 and bad == torch.float16):
            with pytest.raises(TypeError):
                op.process(torch.zeros((2, 128), device=DEV).to(bad), w)
    with pytest.raises(TypeError):
        op.process(torch.zeros((2, 128), dtype=good), w)
    with pytest.raises(capi.LhipError):
        op.process(torch.zeros((2, 96), dtype=good, device=DEV), w)
    with pytest.raises(capi.LhipError):
        op.process(torch.zeros((0, 128), dtype=good, device=DEV), w)
    misaligned = torch.zeros(2 * 128 + 1, dtype=good, device=DEV)[1:].view(2, 128)
    with pytest.raises(capi.LhipError):
        op.process(misaligned, w)
