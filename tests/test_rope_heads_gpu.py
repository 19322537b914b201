"""Rotary embedding and cache append by threads that keep a pair for several heads: head dims around the 256 pairs of a block, fewer and
more heads than a block has side by side, one token and more than a round, positions that run past the cache."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from luminal_amd import capi  # noqa: E402
from oracle import llama_oracle as lo  # noqa: E402

pytestmark = pytest.mark.gpu

DEV, THETA = "cuda:0", 500000.0


@pytest.mark.parametrize("tokens,hq,hkv,hd,pos", [(63, 32, 8, 128, 5), (64, 32, 8, 128, 5), (700, 4, 2, 64, 0), (65, 4, 2, 6, 9), (70, 3, 1, 600, 3),
                                                  (64, 2, 2, 512, 40), (130, 7, 7, 192, 0), (600, 1, 1, 2, 1)])
def test_rope_and_append(tokens, hq, hkv, hd, pos):
    lib = capi.load_library()
    rng = np.random.default_rng(tokens + hd)
    max_seq = pos + tokens - (2 if tokens > 2 else 0)  # the last two of several tokens have no row in the caches
    x = rng.standard_normal((tokens, hq + 2 * hkv, hd)).astype(np.float32)
    qkv = torch.from_numpy(x.copy()).to(DEV)
    kc, vc = (torch.full((hkv, max_seq, hd), 7.0, device=DEV) for _ in range(2))
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    capi.check(lib.lhip_rope_kv_append_f32(qkv.data_ptr(), kc.data_ptr(), vc.data_ptr(), p.data_ptr(), tokens, hq, hkv, hd, max_seq,
                                           THETA, torch.cuda.current_stream().cuda_stream), "rope")
    got, kc, vc = qkv.cpu().numpy(), kc.cpu().numpy(), vc.cpu().numpy()
    want = lo.rope(x[:, :hq + hkv].astype(np.float64), pos, THETA)
    # the angle in f32: pos x a frequency of a few roundings; then two products and their sum
    pair = np.repeat(np.abs(x[:, :hq + hkv, 0::2]) + np.abs(x[:, :hq + hkv, 1::2]), 2, axis=-1)
    assert np.all(np.abs(got[:, :hq + hkv] - want) <= pair * ((pos + tokens) * 2.0 ** -21 + 2.0 ** -21))
    assert np.array_equal(got[:, hq + hkv:], x[:, hq + hkv:])
    n = max_seq - pos
    assert np.array_equal(kc[:, pos:].transpose(1, 0, 2), got[:n, hq:hq + hkv]) and np.array_equal(vc[:, pos:].transpose(1, 0, 2), x[:n, hq + hkv:])
    assert np.all(kc[:, :pos] == 7.0) and np.all(vc[:, :pos] == 7.0)
