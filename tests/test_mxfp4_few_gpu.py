"""The exact expert layer for up to 64 routed rows (mxfp4_moe_few.hip) where its tiles and its walk over K have edges, against the oracle and
stage by stage, with the bars of test_mxfp4_gpu.py."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_mxfp4_gpu import DEV, EXACT, NORM_TOL, check_stages, make_layer, norm_err  # noqa: E402

pytestmark = pytest.mark.gpu


def run(oracle, layer, e, sel, h, seed, poison=()):
    rng = np.random.default_rng(seed)
    t, topk = sel.shape
    bits = oracle.f32_to_bf16_bits((rng.standard_normal((t, h)) * 0.05).astype(np.float32))
    for row in poison:
        bits[row] = 0x7F80  # infinities
    wts = rng.random((t, topk)).astype(np.float32)
    xd = torch.from_numpy(bits.view(np.int16)).to(DEV).view(torch.bfloat16)
    y = layer.process(xd, torch.from_numpy(sel).to(DEV), torch.from_numpy(wts).to(DEV), EXACT).float().cpu().numpy()
    return oracle.bf16_bits_to_f32(bits), wts, y


def rows_of_experts(counts, topk, e):
    """(t, topk) choices in which expert i has counts[i] routed rows, shuffled; -1 and e fill the rest (no expert)."""
    sel = np.concatenate([np.full(c, i) for i, c in enumerate(counts)]).astype(np.int32)
    sel = np.concatenate([sel, np.resize([-1, e], (-sel.size) % topk).astype(np.int32)])
    return np.random.default_rng(sum(counts)).permutation(sel).reshape(-1, topk)


# rows of the experts: around a tile of 16, several tiles, none, all of them one expert's; more experts than lanes; widths: whole and
# ragged chunks of 128, as few and one more than a column block's, every number of chunks a wave holds, one and two segments of them
@pytest.mark.parametrize("counts,topk,h,i", [((15, 16, 17, 0, 1), 1, 160, 96), ((33, 0, 31), 2, 256, 64), ((0, 64, 0, 0), 4, 96, 160), ((5, 7), 2, 3104, 96),
                                             ((3, 1, 2), 1, 128, 3232), ((2, 2), 2, 6240, 6176), ((1, 0, 1, 2), 2, 2880, 3072),
                                             (tuple(int(i % 7 == 0) for i in range(200)), 1, 64, 64), ((9, 3), 2, 992, 320),
                                             ((3, 4, 1), 1, 1312, 1696), ((5, 7), 2, 4160, 7712)])
def test_tiles_of_16_rows(oracle, counts, topk, h, i):
    e = len(counts)
    layer, w_gu, w_dn = make_layer(oracle, e, h, i, seed=h + i)
    sel = rows_of_experts(counts, topk, e)
    xf, wts, y = run(oracle, layer, e, sel, h, seed=e)
    known = (sel >= 0) & (sel < e)
    truth = oracle.moe_forward(xf, w_gu, w_dn, np.where(known, sel, 0), np.where(known, wts, 0.0).astype(np.float32), act_bf16=True)
    assert norm_err(y, truth) < NORM_TOL[EXACT]
    live = np.flatnonzero(known.all(axis=1))
    check_stages(oracle, layer, xf, w_gu, w_dn, sel, wts, y, tokens=live, mode=EXACT)


@pytest.mark.parametrize("t,h,i", [(3, 160, 96), (6, 3104, 96), (1, 96, 3104)])
def test_a_row_s_values_stay_in_it(oracle, t, h, i):
    """A chunk of a ragged K reads nothing of the row behind it: the tokens next to one of infinities stay finite."""
    layer, w_gu, w_dn = make_layer(oracle, 2, h, i, seed=4)
    sel = np.zeros((t, 1), np.int32)
    sel[t // 2] = 1
    clean = run(oracle, layer, 2, sel, h, seed=9)[2]
    dirty = run(oracle, layer, 2, sel, h, seed=9, poison=(t - 1,) if t > 1 else ())[2]
    assert np.isfinite(clean).all() and np.array_equal(clean[:t - 1], dirty[:t - 1])


def test_no_routed_row_names_an_expert(oracle):
    layer, _, _ = make_layer(oracle, 3, 96, 64, seed=2)
    for t in (1, 5):
        assert not run(oracle, layer, 3, np.full((t, 2), 3, np.int32), 96, seed=t)[2].any()
