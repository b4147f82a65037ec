"""The gated product of stacked experts with their weights in its epilogue, against 64 bits: weights from an array or from a table of
the rows' tokens, on the host's or the device's word; rows of one to four tiles, experts that end inside a block's tiles.

Bound: float sums of K products, the gating's few roundings, and half a place of bfloat16 (2^-8)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def case(M, E, f, s, K, seed=0):
    from burn_lm_amd.csrc import ops
    g = torch.Generator(device="cuda").manual_seed(seed + M + E + K)
    I = E * f + s
    x = torch.randn(M, K + 8, generator=g, device="cuda").bfloat16()[:, :K]
    w = (torch.randn(2 * I, K, generator=g, device="cuda") / K ** 0.5).bfloat16()
    return x, w, ops.pack_weight(w, gated=True), torch.full((M, I), float("nan"), dtype=torch.bfloat16, device="cuda"), g


def check(out, x, w, share, E, f):
    I = out.shape[1]
    y, room = x.double() @ w.double().t(), (x.shape[1] + 4) * U * (x.double().abs() @ w.double().abs().t())
    (g, u), (dg, du) = y.chunk(2, 1), room.chunk(2, 1)
    by = share.double()[:, torch.clamp(torch.arange(I, device="cuda") // f, max=E)]
    want = torch.nn.functional.silu(g) * u * by
    slack = (1.1 * dg * u.abs() + du * g.abs() + dg * du + 12 * U * (g * u).abs()) * by.abs()
    assert bool(((out.double() - want).abs() <= slack + 2.0 ** -8 * (want.abs() + slack)).all())
    assert bool((out[by == 0] == 0).all())


@pytest.mark.parametrize("M", [1, 8, 16, 17, 33, 64])
@pytest.mark.parametrize("E,f,s,K", [(4, 8, 0, 64), (3, 24, 16, 520), (16, 512, 0, 2048), (5, 40, 0, 1536)])
def test_weights_from_an_array(M, E, f, s, K):
    from burn_lm_amd.csrc import ops
    x, w, packed, out, g = case(M, E, f, s, K)
    weights = torch.rand(M, E + 1, generator=g, device="cuda") * (torch.rand(M, E + 1, generator=g, device="cuda") < 0.5)
    check(ops.gemv_experts(x, packed, out, E, f, weights=weights), x, w, weights, E, f)
    w[:8] = float("inf")       # an expert nobody chose counts as nothing, whatever it holds
    weights[:, 0] = 0
    packed = ops.pack_weight(w, gated=True)
    assert bool((ops.gemv_experts(x, packed, out, E, f, weights=weights)[:, :8] == 0).all())


@pytest.mark.parametrize("M", [1, 3, 8, 16])
@pytest.mark.parametrize("E,f,top,K", [(16, 512, 4, 2048), (5, 24, 5, 1544), (40, 16, 16, 4096), (7, 8, 1, 64)])
def test_weights_from_a_table(M, E, f, top, K):
    from burn_lm_amd.csrc import ops
    x, w, packed, out, g = case(M, E, f, 0, K, seed=1)
    V = 50
    table = torch.rand(V, E, generator=g, device="cuda").argsort(1)[:, :top].int().contiguous()
    ids = torch.randint(0, V, (M,), generator=g, device="cuda").int()
    ids[-1] = V if M > 1 else 3                   # a token outside the table chooses no expert
    share = torch.empty(M, E + 1, device="cuda")
    ops.moe_table(table, ids, share, E)
    check(ops.gemv_experts(x, packed, out, E, f, table=table, ids=ids), x, w, share, E, f)
    # every second row's token lies in an array on the device
    picked = torch.randint(0, V, (64,), generator=g, device="cuda").int()
    rows = torch.arange(M, device="cuda").int() * 3
    rows[::2] = -1
    source = rows, torch.tensor([picked.data_ptr()], dtype=torch.int64, device="cuda")
    ops.moe_table(table, ids, share, E, source)
    check(ops.gemv_experts(x, packed, out, E, f, table=table, ids=ids, token_source=source), x, w, share, E, f)


def test_what_is_refused():
    from burn_lm_amd.csrc import ops
    x, w, packed, out, g = case(17, 16, 16, 0, 1024)
    table, ids = torch.zeros(9, 4, dtype=torch.int32, device="cuda"), torch.zeros(17, dtype=torch.int32, device="cuda")
    with pytest.raises(ops.KernelError):                     # too many rows for a table
        ops.gemv_experts(x, packed, out, 16, 16, table=table, ids=ids)
    x, w, packed, out, g = case(8, 16, 16, 0, 1024)
    with pytest.raises(ops.KernelError):                     # too many experts a token
        ops.gemv_experts(x, packed, out, 16, 16, table=torch.zeros(9, 17, dtype=torch.int32, device="cuda"), ids=ids)
    with pytest.raises(ops.KernelError):
        ops.gemv_experts(x, packed, out, 16, 16)
    with pytest.raises(ops.KernelError):
        ops.gemv_experts(x, packed, out, 17, 16, weights=torch.zeros(8, 18, device="cuda"))


@pytest.mark.parametrize("M", [16, 17, 32, 33, 64])
@pytest.mark.parametrize("E,f,s,K", [(4, 12, 0, 64), (6, 4, 24, 200), (600, 16, 8, 1024), (300, 32, 0, 512), (3, 104, 8, 1160)])
def test_experts_inside_tiles_and_many_tiles_a_block(M, E, f, s, K):
    """Experts that end inside a tile of eight pairs, and blocks of several tiles, whose weights take turns in shared memory."""
    from burn_lm_amd.csrc import ops
    x, w, packed, out, g = case(M, E, f, s, K, seed=2)
    weights = torch.rand(M, E + 1, generator=g, device="cuda") * (torch.rand(M, E + 1, generator=g, device="cuda") < 0.3)
    check(ops.gemv_experts(x, packed, out, E, f, weights=weights), x, w, weights, E, f)
