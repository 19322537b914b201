"""The bf16 prompt attention over long contexts and at the edges of its pipeline (one tile, an odd and an even number of
tiles in front of and under the causal mask, a partial last tile), for every head shape it is built for."""
import pytest
import torch

from luminal_amd import capi

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("hq,hkv,hd", [(32, 8, 128), (4, 2, 128), (16, 2, 128), (4, 2, 64), (8, 2, 64), (16, 2, 64)])
@pytest.mark.parametrize("S,pos0", [(1, 0), (2, 31), (31, 1), (32, 32), (65, 95), (97, 1951), (2000, 0)])
def test_against_the_f32_kernel(hq, hkv, hd, S, pos0):
    """|y - t| < 2e-2 sum_j p_j |v_j| (+ the same for the f32 kernel's own 1e-5): three roundings to bf16 (V, the weights,
    the result) bound the error by 3 * 2^-8 of that sum, those of q and K add the error of a score.  t comes from the f32
    matrix-core kernel, the sum from the same kernel over |V|."""
    lib = capi.load_library()
    gen = torch.Generator(device=DEV).manual_seed(S * 7 + pos0 + hq)
    room = pos0 + S + 5
    kc, vc = (torch.randn((hkv, room, hd), device=DEV, generator=gen) for _ in range(2))
    # rows that no query may see: they must not reach the result
    kc[:, pos0 + S:] = float("nan")
    vc[:, pos0 + S:] = float("nan")
    qkv = torch.randn((S, (hq + 2 * hkv) * hd), device=DEV, generator=gen)
    pos = torch.tensor([pos0], dtype=torch.int32, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    dims = (pos.data_ptr(), S, hq, hkv, hd, room, stream)
    got = torch.full((S, hq * hd), float("nan"), device=DEV, dtype=torch.bfloat16)
    exact, scale = torch.empty((S, hq * hd), device=DEV), torch.empty((S, hq * hd), device=DEV)
    v_abs = vc.abs().nan_to_num(0.0)
    v_fin, k_fin = vc.nan_to_num(0.0), kc.nan_to_num(0.0)
    assert lib.lhip_attention_bf16(qkv.data_ptr(), kc.data_ptr(), vc.data_ptr(), got.data_ptr(), *dims) == 0
    assert lib.lhip_attention_f32(qkv.data_ptr(), k_fin.data_ptr(), v_fin.data_ptr(), exact.data_ptr(), *dims) == 0
    assert lib.lhip_attention_f32(qkv.data_ptr(), k_fin.data_ptr(), v_abs.data_ptr(), scale.data_ptr(), *dims) == 0
    worst = float(((got.float() - exact).abs() / scale).max())
    assert worst < 2e-2 + 1e-5, worst
