"""Decode attention over a cache of at most 512 positions, which is one launch: bit for bit the two launches of a longer cache that
holds the same keys and values, at every edge of its ranges, and the same rows appended to the caches."""
import pytest
import torch

from luminal_amd import capi

DEV = "cuda:0"
# (query heads, KV heads, head dim, positions): 32 ranges of up to 16 keys, 16 ranges, 32 ranges of fewer keys, one query head a KV head
SHAPES = [(32, 8, 128, 512), (32, 16, 64, 256), (64, 8, 64, 300), (8, 8, 128, 512)]


def decode(lib, qkv, k, v, pos, hq, hkv, hd, max_seq):
    out = torch.full((hq * hd,), float("nan"), device=DEV)
    ws = torch.full((lib.lhip_attention_decode_workspace_nbytes(hq, hkv, hd),), 255, dtype=torch.uint8, device=DEV)
    p = torch.tensor([pos], dtype=torch.int32, device=DEV)
    capi.check(lib.lhip_attention_decode_f32(qkv.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), p.data_ptr(), hq, hkv, hd,
                                             max_seq, 500000.0, ws.data_ptr(), torch.cuda.current_stream().cuda_stream), "decode")
    torch.cuda.synchronize()
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,hd,short", SHAPES)
def test_one_launch_gives_the_bits_of_two(hq, hkv, hd, short):
    lib = capi.load_library()
    gen = torch.Generator(device=DEV).manual_seed(hq + hd)
    long = 1024
    k_long, v_long = (torch.randn((hkv, long, hd), device=DEV, generator=gen) for _ in range(2))
    for pos in (0, 1, 14, 15, 16, 31, 32, 33, 100, 255, short // 2 + 1, short - 2, short - 1):
        if pos >= short:
            continue
        qkv = torch.randn(((hq + 2 * hkv) * hd,), device=DEV, generator=gen) * 3.0
        ks, vs = (t[:, :short].contiguous() for t in (k_long, v_long))
        kl, vl = k_long.clone(), v_long.clone()
        one, two = decode(lib, qkv, ks, vs, pos, hq, hkv, hd, short), decode(lib, qkv, kl, vl, pos, hq, hkv, hd, long)
        assert torch.equal(one.view(torch.int32), two.view(torch.int32)), pos
        assert torch.equal(ks, kl[:, :short]) and torch.equal(vs, vl[:, :short]) and not torch.equal(kl, k_long), pos


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,hd,short", SHAPES)
def test_rows_not_written_yet_and_an_infinite_value_stay_where_they_belong(hq, hkv, hd, short):
    """From the new position on the caches hold NaN and the new value has infinities, at positions that a range begins with (all below
    the number of ranges, multiples of a range's keys) and others: neither reaches a slot behind the range's end, by either form."""
    lib = capi.load_library()
    gen = torch.Generator(device=DEV).manual_seed(hq + hd + 1)
    long = 1024
    keys, values = (torch.randn((hkv, long, hd), device=DEV, generator=gen) for _ in range(2))
    for pos in (0, 1, 2, 15, 30, 31, 32, 33, 40, 96, 97, 200, 252, 300, short - 1):
        if pos >= short:
            continue
        qkv = torch.randn(((hq + 2 * hkv) * hd,), device=DEV, generator=gen)
        kc, vc = keys.clone(), values.clone()
        clean = decode(lib, qkv, kc, vc, pos, hq, hkv, hd, long).view(hq, hd)
        qkv.view(-1, hd)[hq + hkv:, 3::8] = float("inf")
        for max_seq in (short, long):
            kc, vc = (t[:, :max_seq].clone() for t in (keys, values))
            kc[:, pos:] = vc[:, pos:] = float("nan")
            out = decode(lib, qkv, kc, vc, pos, hq, hkv, hd, max_seq).view(hq, hd)
            assert bool((out[:, 3::8] == float("inf")).all()), (pos, max_seq)
            rest = [c for c in range(hd) if c % 8 != 3]
            assert torch.equal(out[:, rest].view(torch.int32), clean[:, rest].view(torch.int32)), (pos, max_seq)
