"""The float32 products on the matrix cores alone: every tile, the edges of tiles, remainders of K, groups of K, the gating,
rows that are longer than what is multiplied; and the runtime's choice among them over the forms that it accepts.

The bound on an element's error is that of a sum of K products in any order with one rounding per product and addition:
(K + 2) 2^-24 times the sum of the products' sizes (and a few roundings more for the gating)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def operands(M, N, K, pad=0, seed=0):
    g = torch.Generator().manual_seed(seed)
    whole = torch.full((M, K + pad), float("nan"))
    whole[:, :K] = torch.randn(M, K, generator=g)
    return whole.cuda()[:, :K], torch.randn(N, K, generator=g).cuda()


def check(got, x, w, gated=False):
    x64, w64 = x.double(), w.double()
    want, room = x64 @ w64.t(), (x.shape[1] + 2) * EPS * (x64.abs() @ w64.abs().t())
    if gated:
        g, u = want.chunk(2, -1)
        dg, du = room.chunk(2, -1)
        want = torch.nn.functional.silu(g) * u
        room = 1.1 * dg * u.abs() + du * g.abs() + dg * du + 8 * EPS * want.abs()     # |silu'| < 1.1, |silu(g)| <= |g|
    assert bool(((got.double() - want).abs() <= room + 1e-30).all()), float(((got.double() - want).abs() / (room + 1e-30)).max())


@pytest.mark.parametrize("tile", [(128, 128), (128, 64), (64, 128), (64, 64)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 4), (17, 33, 28), (63, 64, 32), (64, 65, 36), (65, 130, 160), (129, 127, 260), (257, 515, 96)])
def test_many_rows(tile, M, N, K):
    from burn_lm_amd.csrc import ops
    x, w = operands(M, N, K, pad=4 * (M % 3))
    check(ops.gemm_f32(x, w, torch.full((M, N), float("nan"), device="cuda"), tile=tile), x, w)
    for groups in (2, 3, 8):
        check(ops.gemm_f32(x, w, torch.full((groups, M, N), float("nan"), device="cuda"), tile=tile).sum(0), x, w)


@pytest.mark.parametrize("tile", [(128, 128), (64, 128)])
@pytest.mark.parametrize("M,I,K", [(17, 8, 28), (64, 64, 32), (65, 65, 36), (129, 200, 260)])
def test_many_rows_gated(tile, M, I, K):
    from burn_lm_amd.csrc import ops
    x, w = operands(M, 2 * I, K, pad=4)
    check(ops.gemm_f32(x, w, torch.full((M, I), float("nan"), device="cuda"), gated=True, tile=tile), x, w, gated=True)


@pytest.mark.parametrize("M", [1, 4, 5, 15, 16])
@pytest.mark.parametrize("N,K", [(1, 4), (16, 16), (17, 20), (100, 512), (33, 516), (48, 2048), (2048, 2044)])
def test_few_rows(M, N, K):
    from burn_lm_amd.csrc import ops
    x, w = operands(M, N, K, pad=4 * (M % 2))
    packed = ops.pack_weight(w)
    for groups in (1, 2, 3):
        out = torch.full((groups, M, N), float("nan"), device="cuda")
        check((ops.gemv_f32(x, packed, out, K)).sum(0), x, w)
    wide = torch.full((M, N + 3), float("nan"), device="cuda")
    check(ops.gemv_f32(x, packed, wide[:, :N], K), x, w)
    assert bool(wide[:, N:].isnan().all())


@pytest.mark.parametrize("M", [1, 8, 16])
@pytest.mark.parametrize("N,K,groups", [(4112, 2048, 1), (8200, 2048, 1), (8200, 2048, 3), (8209, 512, 1), (16400, 260, 2), (4099, 1000, 2)])
def test_few_rows_of_many_columns(M, N, K, groups):
    """Blocks that walk several column tiles, the last one fewer: weights asked for ahead across tiles, the same shared memory for
    every tile's sums."""
    from burn_lm_amd.csrc import ops
    blocks, _ = ops.gemv_f32_geometry(M, N, K, groups)
    tiles = -(-N // 16)
    assert blocks // groups < tiles           # so some block has more than one
    x, w = operands(M, N, K, seed=N)
    out = torch.full((groups, M, N), float("nan"), device="cuda")
    check(ops.gemv_f32(x, ops.pack_weight(w), out, K).sum(0), x, w)


@pytest.mark.parametrize("M,I,K", [(1, 8, 4), (3, 24, 100), (8, 72, 516), (16, 256, 2048)])
def test_few_rows_gated(M, I, K):
    from burn_lm_amd.csrc import ops
    x, w = operands(M, 2 * I, K)
    check(ops.gemv_f32(x, ops.pack_weight(w, gated=True), torch.full((M, I), float("nan"), device="cuda"), K, gated=True), x, w, gated=True)


@pytest.mark.parametrize("K,at,groups", [(520, 516, 1), (64, 63, 1), (2048, 43 * 16, 3), (2048, 0, 3), (516, 512, 2)])
@pytest.mark.parametrize("M", [1, 8, 16])
def test_an_infinite_weight_stays_infinite(M, K, at, groups):
    """Wavefronts whose stretch of K is shorter than the others' have steps without weights: these add zeros, whatever the
    matrix holds elsewhere."""
    from burn_lm_amd.csrc import ops
    x, w = operands(M, 33, K)
    x = x.abs() + 0.5
    w[3, at], w[20, at] = float("inf"), float("-inf")
    got = ops.gemv_f32(x, ops.pack_weight(w), torch.empty(groups, M, 33, device="cuda"), K).sum(0)
    assert bool((got[:, 3] == float("inf")).all()) and bool((got[:, 20] == float("-inf")).all())
    others = [n for n in range(33) if n not in (3, 20)]
    check(got[:, others], x, w[others])


@pytest.mark.parametrize("M,I,K", [(1, 4104, 2048), (8, 4136, 512), (16, 4104, 2048)])
def test_few_rows_of_many_pairs(M, I, K):
    from burn_lm_amd.csrc import ops
    assert ops.gemv_f32_geometry(M, 2 * I, K)[0] < I // 8
    x, w = operands(M, 2 * I, K, seed=I)
    check(ops.gemv_f32(x, ops.pack_weight(w, gated=True), torch.full((M, I), float("nan"), device="cuda"), K, gated=True), x, w, gated=True)


def test_refused():
    from burn_lm_amd.csrc import ops
    x, w = operands(17, 32, 2052)
    out = torch.empty(17, 32, device="cuda")
    with pytest.raises(ops.KernelError):
        ops.gemv_f32(x, ops.pack_weight(w), out, 2052)                        # 17 rows
    with pytest.raises(ops.KernelError):
        ops.gemv_f32(x[:8], ops.pack_weight(w), out[:8], 2052)                # more than a group's stretch
    with pytest.raises(ops.KernelError):
        ops.gemm_f32(x[:, 1:], w[:, 1:].contiguous(), out)                    # rows at odd addresses
    assert not ops.f32_rows(x[:, 1:], w) and not ops.f32_rows(x.t(), w) and not ops.f32_rows(x.bfloat16(), w)


@pytest.mark.parametrize("K", [64, 70, 2048, 2052, 4100])
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 70])
def test_runtime_takes_every_form(M, K):
    """The choice of kernel against 64 bits: weights that were bound, plain ones, results that come as planes or go into a given
    tensor, rows with a stride, sizes that are no multiples of four (the older kernels), gated and not."""
    from burn_lm_amd.engine.runtime import Runtime
    rt = Runtime(torch.float32, "cuda:0")
    x, w = operands(M, 48, K, pad=0 if K % 4 else 8)
    for weight in (rt.weight(w), w):
        check(rt.linear(x, weight), x, w)
        got = rt.linear(x, weight, partials=True)
        check(got.sum(0) if got.dim() == 3 else got, x, w)
        given = torch.full((M, 50), float("nan"), device="cuda")
        check(rt.linear(x, weight, out=given[:, :48]), x, w)
        assert bool(given[:, 48:].isnan().all())
    check(rt.gated_linear(x, rt.weight(w, gated=True)), x, w, gated=True)
    check(rt.gated_linear(x, w), x, w, gated=True)


@pytest.mark.parametrize("why", ["little is free", "the model is large", "the allocation fails"])
def test_no_room_for_packed_copies(why, monkeypatch):
    """Where the matrices do not fit the device's memory a second time, products of few rows read them as they are: nothing is
    refused, and the matrix keeps that form."""
    from burn_lm_amd.csrc import ops
    from burn_lm_amd.engine.runtime import Runtime
    rt = Runtime(torch.float32, "cuda:0")
    size = 4 * 2048 * 2048
    if why == "the allocation fails":
        def fails(w, gated=False):
            raise torch.cuda.OutOfMemoryError("out of memory")
        monkeypatch.setattr(ops, "pack_weight", fails)
    else:
        free, total = (0, 64 * size) if why == "little is free" else (60 * size, 64 * size)
        held = torch.cuda.memory_reserved() - torch.cuda.memory_allocated()
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda *a: (free - held, total))
    made = [rt.weight(operands(1, 2048, 2048, seed=i)[1], gated=i == 1) for i in range(10)]
    for M in (1, 8, 9, 16):
        x = operands(M, 1, 2048)[0]
        for i, w in enumerate(made):
            check((rt.gated_linear if w.gated else rt.linear)(x, w), x, w.w, gated=w.gated)
    packed = [w.is_packed for w in made]
    assert packed == ([True] * 8 + [False] * 2 if why == "the model is large" else [False] * 10)
    if why == "the model is large":      # memory that is given back serves another
        made[0].drop_packed()
        assert rt.weight(made[9].w).packed is not None


def test_plan_keeps_its_bounds():
    from burn_lm_amd.engine.runtime import f32_plan
    for M in (9, 64, 65, 1000):
        for N in (1, 64, 5000):
            for K in (4, 130, 8192):
                tile, groups, us = f32_plan(M, N, K, 256, planes=True)
                assert groups == 1 or K // groups >= 128
                assert f32_plan(M, N, K, 256)[1] == 1 and f32_plan(M, N, K, 256, gated=True)[0][1] == 128 and us > 0


def test_plan_is_made_once():
    """The same sizes again take the plan that was made for them, within a bounded number of plans."""
    from burn_lm_amd.engine.runtime import f32_plan
    assert f32_plan(777, 2048, 8192, 256, planes=True) is f32_plan(777, 2048, 8192, 256, planes=True)
    assert f32_plan(777, 2048, 8192, 256) is not f32_plan(777, 2048, 8192, 256, planes=True)
    assert f32_plan.cache_info().maxsize is not None


@pytest.mark.parametrize("M,K,nh,nkv,hd", [(1, 64, 2, 1, 16), (3, 36, 3, 1, 6), (8, 2048, 32, 8, 64), (16, 520, 5, 5, 34), (7, 272, 1, 1, 128)])
def test_projection_with_rotation_and_pages(M, K, nh, nkv, hd):
    """Up to 16 rows: the fused kernel's queries and pages are those of the product followed by the rotation kernel (a rotation is two
    products and a sum: an ulp of the larger one apart at most); a padding row writes no page, heads may end inside a tile of columns."""
    from burn_lm_amd.csrc import ops
    from burn_lm_amd.engine.runtime import Runtime
    rt = Runtime(torch.float32, "cuda:0")
    g = torch.Generator().manual_seed(M + K)
    N, page = (nh + 2 * nkv) * hd, 64
    x, w = torch.randn(M, K, generator=g).cuda(), rt.weight((torch.randn(N, K, generator=g) * K ** -0.5).cuda())
    pos = torch.tensor([(37 * i + 5) % 250 for i in range(M)], dtype=torch.int32).cuda()
    seq = torch.arange(M, dtype=torch.int32)
    if M > 2:
        seq[1] = -1
    seq, table = seq.cuda(), torch.randperm(4 * M, generator=g).view(M, 4).int().cuda()
    cs = torch.randn(256, hd // 2, 2, generator=g).cuda()
    got = []
    for fused in (True, False):
        k, v = (torch.full((4 * M, nkv, *s), 9.0, device="cuda") for s in ((page, hd), (hd, page)))
        for store in (False, True):
            if fused:
                packed = rt.f32_qkv_packed(x, w, M, N, K)
                out = ops.gemv_f32_qkv_rope(x, packed, torch.full((M, N), 7.0, device="cuda"), pos, seq, table, cs, k, v, page, nh, nkv, hd, write_kv=store)
                assert bool((out[:, nh * hd:] == 7).all())
            else:
                out = rt.linear(x, w)
                ops.rope_kv_write(out, pos, seq, table, cs, k, v, page, nh, nkv, hd, 0, write_kv=store)
            assert store or bool((k == 9).all() and (v == 9).all())
        got.append((out[:, :nh * hd][seq >= 0], k, v))
    for a, b in zip(*got):
        assert torch.allclose(a, b, rtol=2.0 ** -21, atol=2.0 ** -20)
    assert torch.equal(got[0][2], got[1][2])
