"""The rotation behind the packed q/k/v product, bit by bit: a lane's own product joins its partner's, which is rounded, in one rounding."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("M,K", [(1, 64), (8, 64), (8, 2048), (5, 4096), (16, 512), (17, 512), (33, 2048), (64, 264)])
def test_turned_pairs(M, K, scaled):
    """Rows of a single one pick columns of the weights, so that the products are exact, and the angles are such that one lane of every pair is
    what is left of two products that cancel: all of it is the rounding of one of them."""
    from burn_lm_amd.csrc import ops
    if scaled and (M > 8 or K & (K - 1)):
        pytest.skip("unscaled rows are eight at most; their factor is one for widths of a power of two")
    g = torch.Generator().manual_seed(M + K)
    nh, nkv, hd, page = 2, 1, 32, 64
    head = ((torch.rand(hd, K, generator=g) + 0.5) * torch.randn(hd, K, generator=g).sign()).bfloat16()
    x = torch.eye(M, K).bfloat16()
    u, w = head[0::2, :M].t().double(), head[1::2, :M].t().double()          # [row, pair]
    cos = torch.rand(M, hd // 2, generator=g) + 0.5
    even = torch.arange(hd // 2) % 2 == 0
    sin = torch.where(even, cos.double() * u / w, -cos.double() * w / u).float()
    rounded = lambda a: (a * sin.double()).float().double()
    want = torch.stack((u * cos.double() - rounded(w), w * cos.double() + rounded(u)), -1).float().bfloat16().reshape(M, hd)
    assert bool((want != 0).any())

    out = torch.zeros(M, (nh + 2 * nkv) * hd, dtype=torch.bfloat16, device="cuda")
    k, v = (torch.zeros(M, nkv, *s, dtype=torch.bfloat16, device="cuda") for s in ((page, hd), (hd, page)))
    rows = torch.arange(M, dtype=torch.int32, device="cuda")
    scale = (torch.full((M, 4), K / 4.0, device="cuda"), 0.0) if scaled else None
    ops.gemv_qkv_rope(x.cuda(), ops.pack_weight(head.repeat(nh + 2 * nkv, 1).cuda()), out, rows % page, rows, rows.view(M, 1),
                      torch.stack((cos, sin), -1).cuda(), k, v, page, nh, nkv, hd, 0, scale=scale)
    at = torch.arange(M)
    for got in (out[:, :hd].cpu(), out[:, hd:2 * hd].cpu(), k.cpu()[at, 0, at % page]):
        assert torch.equal(got, want)
    assert torch.equal(v.cpu()[at, 0, :, at % page], head[:, :M].t())
