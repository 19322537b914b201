"""Decode attention where its key ranges change how they are read: up to 32 keys through the caches and from 33 past them,
and ranges around one tile of 64 keys and of several, against rotary + append + softmax(QK)V in f64."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from luminal_amd import capi  # noqa: E402
from oracle import llama_oracle as lo  # noqa: E402

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


# keys per range of a launch with 256 / kv_heads ranges; the last range of each is shorter by the one key that is missing
@pytest.mark.parametrize("hq,hkv,hd", [(32, 8, 128), (16, 8, 64)])
@pytest.mark.parametrize("range_keys", [31, 32, 33, 64, 65, 130])
def test_lengths_of_a_key_range(hq, hkv, hd, range_keys):
    lib = capi.load_library()
    rng = np.random.default_rng(range_keys)
    p = range_keys * (256 // hkv) - 2
    max_seq = p + 5
    g = hq // hkv
    kc, vc = (torch.from_numpy(rng.standard_normal((hkv, max_seq, hd)).astype(np.float32)).to(DEV) for _ in range(2))
    qkv = (2.0 * rng.standard_normal((hq + 2 * hkv, hd))).astype(np.float32)
    ws = torch.full((lib.lhip_attention_decode_workspace_nbytes(hq, hkv, hd),), 0xFF, dtype=torch.uint8, device=DEV)
    out = torch.empty((hq, hd), device=DEV)
    pos = torch.tensor([p], dtype=torch.int32, device=DEV)
    qd = torch.from_numpy(qkv).to(DEV)
    capi.check(lib.lhip_attention_decode_f32(qd.data_ptr(), kc.data_ptr(), vc.data_ptr(), out.data_ptr(), pos.data_ptr(), hq, hkv,
                                             hd, max_seq, 500000.0, ws.data_ptr(), torch.cuda.current_stream().cuda_stream), "decode")
    q = lo.rope(qkv[None, :hq].astype(np.float64), p, 500000.0)[0]
    k_new = lo.rope(qkv[None, hq:hq + hkv].astype(np.float64), p, 500000.0)[0]
    keys, values = kc.cpu().numpy().astype(np.float64)[:, :p + 1], vc.cpu().numpy().astype(np.float64)[:, :p + 1]
    keys[:, p], values[:, p] = k_new, qkv[hq + hkv:]
    want = np.empty((hq, hd))
    for h in range(hq):
        sc = keys[h // g] @ q[h] / np.sqrt(hd)
        w = np.exp(sc - sc.max())
        want[h] = (w / w.sum()) @ values[h // g]
    # f32 soft-max against the scale of the output, and the f32 rotary angle: half an ulp of p turns q and k by p * 2^-24
    # rad, which moves a score by that times |q||k| / sqrt(hd) (about 25 here)
    err = np.max(np.abs(out.cpu().numpy() - want)) / np.sqrt(np.mean(want * want))
    assert err < 1e-4 + 25 * p * 2.0 ** -24, err
