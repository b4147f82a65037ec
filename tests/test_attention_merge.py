"""Attention of single tokens in pieces, where four dims a thread add the pieces up: more dims than the block has threads, two head tiles with
few heads in the last, none to a full trip's and more pieces, pieces without keys, a token of no sequence."""
import pytest
import torch

from test_attention_f32 import PAGE, case, check

pytestmark = pytest.mark.gpu
LENS = [2200, 1, 130, 64]


def run(op, q, table, kc, vc, nh, nkv, hd, window, splits):
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    out = torch.full((len(LENS) + 1, nh * hd), 7.0, device="cuda", dtype=q.dtype)
    op(q, q.stride(0), out, i32([n - 1 for n in LENS] + [0]), i32([0, 1, 2, 3, -1]), table.cuda(), kc.to(q.dtype).cuda(), vc.to(q.dtype).cuda(), PAGE, nh, nkv,
       hd, hd ** -0.5, window, splits)
    out = out.cpu().reshape(-1, nh, hd)
    assert bool((out[-1] == 0).all())
    return out


@pytest.mark.parametrize("splits", [1, 2, 16, 17, 33])
@pytest.mark.parametrize("window", [0, 100])
@pytest.mark.parametrize("nh,nkv,hd", [(16, 2, 64), (5, 1, 64), (17, 1, 48), (18, 2, 128), (3, 1, 96), (40, 2, 16)])
def test_pieces(nh, nkv, hd, window, splits):
    """float32 within the bound of its sums; bfloat16 within one rounding of the weights and one of the result, 2^-9 of the largest value each."""
    from burn_lm_amd.csrc import ops
    table, keys, values, kc, vc = case(LENS, nkv, hd, 11)
    q = torch.randn(len(LENS) + 1, nh * hd, generator=torch.Generator().manual_seed(12))
    for _ in range(2):         # the second call finds the counters as the first left them
        got = run(ops.attn_decode_f32, q.cuda(), table, kc, vc, nh, nkv, hd, window, splits)
    for b, n in enumerate(LENS):
        check(got[b], q[b].reshape(nh, hd), keys[b], values[b], n - 1, hd ** -0.5, window, nh // nkv)
    for _ in range(2):
        got = run(ops.attn_decode, q.bfloat16().cuda(), table, kc, vc, nh, nkv, hd, window, splits)
    for b, n in enumerate(LENS):
        k, v = (t[max(0, n - window) if window else 0:].bfloat16().double().repeat_interleave(nh // nkv, 1) for t in (keys[b], values[b]))
        w = torch.softmax(torch.einsum("hd,nhd->hn", q[b].bfloat16().double().reshape(nh, hd), k) * hd ** -0.5, -1)
        assert bool(((got[b].double() - torch.einsum("hn,nhd->hd", w, v)).abs() <= 2.0 ** -8 * v.abs().amax((0, 2))[:, None]).all())
