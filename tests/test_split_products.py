"""The float32 products by three bfloat16 parts of every float (gemm_split): the parts, every tile, edges of tiles, groups of K, gating,
values that have no parts, the error beside the float instructions', and the runtime's choice.

The bound on an element's error is that of a sum of K products in any order with one rounding per product and addition, as for the float
instructions (test_f32_products): the products of parts that are left out are below 2^-26 of a product."""
import pytest
import torch

from test_f32_products import check, operands

TILES = [(128, 256), (128, 128), (64, 256), (64, 128)]
INF, NAN = float("inf"), float("nan")


def whole_again(parts, M, K):
    """The floats that the parts add up to (in 64 bits)."""
    p = parts.double().sum(2).reshape(-1, K // 32, 4, 16, 2, 4)              # [row tile, step, quarter, row, half, element]
    return p.permute(0, 3, 1, 4, 2, 5).reshape(-1, K)[:M]                    # element 16 half + 4 quarter + e of a step


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,pad", [(1, 32, 0), (16, 64, 4), (17, 160, 0), (45, 416, 8)])
def test_parts_are_the_float(M, K, pad):
    from burn_lm_amd.csrc import ops
    x, _ = operands(M, 1, K, pad)
    x.mul_(torch.exp2(torch.randint(-60, 60, (M, K), generator=torch.Generator().manual_seed(1)).float().cuda()))
    x[0, 0], x[-1, -1], x[M // 2, 3] = 0.0, torch.finfo(torch.float32).max, -torch.finfo(torch.float32).max
    parts = ops.split_rows(x)
    assert torch.equal(whole_again(parts, M, K), x.double())
    rest = parts.reshape(-1, K // 32, 3, 4, 16, 8)[-1, :, :, :, M % 16 or 16:]
    assert bool((rest == 0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (17, 48, 256), (64, 128, 384), (65, 144, 128), (128, 272, 640), (129, 256, 256), (300, 528, 512)])
def test_tiles(tile, M, N, K):
    from burn_lm_amd.csrc import ops
    x, w = operands(M, N, K, pad=4 * (M % 3))
    parts = ops.split_rows(x)
    wide = torch.full((M, N + 4), NAN, device="cuda")
    check(ops.gemm_split(parts, w, wide[:, :N], tile=tile), x, w)
    assert bool(wide[:, N:].isnan().all())
    for groups in (2, 5):
        if (groups - 1) * -(-(K // 128) // groups) < K // 128:
            check(ops.gemm_split(parts, w, torch.full((groups, M, N), NAN, device="cuda"), tile=tile).sum(0), x, w)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [(128, 256), (64, 256)])
@pytest.mark.parametrize("M,I,K", [(17, 16, 128), (64, 128, 384), (130, 144, 256), (129, 400, 512)])
def test_gated(tile, M, I, K):
    from burn_lm_amd.csrc import ops
    x, w = operands(M, 2 * I, K, pad=4)
    check(ops.gemm_split(ops.split_rows(x), w, torch.full((M, I), NAN, device="cuda"), gated=True, tile=tile), x, w, gated=True)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [(128, 256), (64, 256)])
@pytest.mark.parametrize("M,I,K", [(17, 32, 128), (64, 128, 384), (130, 160, 256), (129, 416, 512)])
def test_gated_results_as_parts(tile, M, I, K):
    """The parts add up to those of the results that the same product stores, also of what is no finite number; rows behind the last are zero."""
    from burn_lm_amd.csrc import ops
    x, w = operands(M, 2 * I, K)
    x[M // 2, 5], x[M - 1, 9], w[3, 7], w[I + 5, 8] = INF, NAN, -INF, torch.finfo(torch.float32).max
    rows = ops.split_rows(x)
    want = ops.split_rows(ops.gemm_split(rows, w, torch.empty(M, I, device="cuda"), gated=True, tile=tile))
    parts = ops.gemm_split_parts(rows, w, M, tile=tile)
    assert torch.equal(*(torch.nan_to_num(whole_again(p, M, I), 7.0, 1e300, -1e300) for p in (parts, want)))
    assert bool((parts.reshape(-1, I // 32, 3, 4, 16, 8)[-1, :, :, :, M % 16 or 16:] == 0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M", [17, 100, 500])
@pytest.mark.parametrize("I,K,N", [(1024, 512, 512), (4096, 1024, 1024), (416, 512, 256), (1000, 256, 128)])
def test_pair(M, I, K, N):
    """Both products of a feed-forward in one call: what they are apart, within the second one's own bound on either order of its sums."""
    from burn_lm_amd.engine.runtime import Runtime
    rt = Runtime(torch.float32, "cuda:0")
    x, w = operands(M, 2 * I, K, pad=4)
    _, down = operands(1, N, I)
    got = rt.gated_pair(x, rt.weight(w, gated=True), rt.weight(down))
    mid = rt.gated_linear(x, w)
    check(got.sum(0) if got.dim() == 3 else got, mid, down)


@pytest.mark.gpu
@pytest.mark.parametrize("M,I,K,N", [(331, 4096, 1024, 1024), (200, 4992, 1152, 1152), (497, 4992, 1152, 1152), (1001, 2176, 1024, 512)])
def test_pair_by_parts(M, I, K, N, monkeypatch):
    """Sizes at which the first product does leave parts, rows that end inside a tile and inner sizes of an odd number of chunks among them: as above,
    also with a row of no numbers, which is one in the result and none of the others."""
    from burn_lm_amd.csrc import ops
    from burn_lm_amd.engine.runtime import Runtime
    left, parts = [], ops.gemm_split_parts
    monkeypatch.setattr(ops, "gemm_split_parts", lambda *a, **k: left.append(1) or parts(*a, **k))
    rt = Runtime(torch.float32, "cuda:0")
    x, w = operands(M, 2 * I, K, pad=4)
    _, down = operands(1, N, I)
    x[M - 2] = NAN
    got = rt.gated_pair(x, rt.weight(w, gated=True), rt.weight(down))
    assert left == [1]
    got, mid = got.sum(0) if got.dim() == 3 else got, rt.gated_linear(x, w)
    assert bool(got[M - 2].isnan().all())
    rest = torch.arange(M, device="cuda") != M - 2
    check(got[rest], mid[rest], down)


@pytest.mark.gpu
@pytest.mark.parametrize("K,groups", [(2048, 1), (2048, 4), (8192, 1), (8192, 4)])
@pytest.mark.parametrize("spread", [0.0, 2.0])
def test_no_further_from_64_bits(K, groups, spread):
    """2-norm of the error, normal values and ones that spread over some powers of ten: no larger than the float instructions'."""
    from burn_lm_amd.csrc import ops
    x, w = operands(300, 512, K, seed=K)
    g = torch.Generator().manual_seed(2)
    x, w = (t * torch.exp(spread * torch.randn(t.shape, generator=g)).cuda() for t in (x, w))
    want = x.double() @ w.double().t()
    err = lambda y: float((y.double() - want).norm() / want.norm())
    out = lambda: torch.empty(groups, 300, 512, device="cuda")
    theirs = err(ops.gemm_f32(x, w, out()).sum(0))
    for tile in TILES:
        assert err(ops.gemm_split(ops.split_rows(x), w, out(), tile=tile).sum(0)) <= theirs


@pytest.mark.gpu
@pytest.mark.parametrize("K,groups", [(128, 1), (256, 1), (384, 1), (640, 1), (1152, 1), (2560, 4), (3072, 8), (4224, 7), (11008, 8)])
@pytest.mark.parametrize("positive", [False, True])
def test_no_offset(K, groups, positive):
    """What the matrix instruction cuts cancels in every group of K, odd numbers of chunks among them (4,224: of five, and of three in the last):
    the mean of the errors is what so many independent ones leave, within five standard deviations, and their 2-norm no larger than the float
    instructions'."""
    from burn_lm_amd.csrc import ops
    M, N = 300, 512
    x, w = operands(M, N, K, seed=K + 1)
    if positive:
        x, w = x.abs(), w.abs()
    want = x.double() @ w.double().t()
    out = lambda: torch.empty(groups, M, N, device="cuda")
    theirs = (ops.gemm_f32(x, w, out()).sum(0).double() - want).norm()
    for tile in TILES:
        planes = ops.gemm_split(ops.split_rows(x), w, out(), tile=tile)
        err = planes.double().sum(0) - want                                  # (without the roundings of the planes' sum)
        assert abs(float(err.mean())) <= 5 * float(err.std()) / (M * N) ** 0.5
        assert (planes.sum(0).double() - want).norm() <= theirs


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
def test_values_without_parts(tile):
    """Infinities, NaN and floats that round to an infinity as a bfloat16, in rows and in weights: what a sum of float products gives."""
    from burn_lm_amd.csrc import ops
    huge = torch.finfo(torch.float32).max
    x, w = operands(70, 160, 256)
    w[5, 7] = 0.0
    w.mul_(2.0 ** -12)
    for m, k, v in ((1, 7, INF), (2, 9, -INF), (3, 200, NAN), (4, 0, huge), (66, 255, -huge), (68, 30, INF)):
        x[m, k] = v
    x[68, 31] = -INF
    w[20, 40], w[30, 41], w[159, 42], w[40, 50] = INF, -INF, NAN, huge
    x[:, 50] = x[:, 50].sign() * 2.0 ** -20
    want = (x.double() @ w.double().t())
    for groups in (1, 2):
        got = ops.gemm_split(ops.split_rows(x), w, torch.empty(groups, 70, 160, device="cuda"), tile=tile).sum(0)
        assert torch.equal(got.isnan(), want.isnan())
        assert torch.equal(got.isposinf(), want.isposinf()) and torch.equal(got.isneginf(), want.isneginf())
        size = x.double().abs() @ w.double().abs().t()
        fine = want.isfinite() & size.isfinite()
        assert bool(((got.double() - want).abs()[fine] <= 258 * 2.0 ** -24 * size[fine]).all())
    if tile[1] == 256:
        gate = ops.gemm_split(ops.split_rows(x), w, torch.empty(70, 80, device="cuda"), gated=True, tile=tile)
        with_inf = torch.nn.functional.silu(want[:, :80]) * want[:, 80:]
        assert torch.equal(gate.isnan(), with_inf.isnan()) and torch.equal(gate.isposinf(), with_inf.float().isposinf())
        assert torch.equal(gate.isneginf(), with_inf.float().isneginf())


def sprinkled(M, N, K, what):
    """Operands with values that are no finite number (or round to none as a bfloat16) in the places that `what` names."""
    x, w = operands(M, N, K, seed=len(what))
    w.mul_(2.0 ** -12)
    g = torch.Generator().manual_seed(7)
    at = lambda n: torch.randint(0, K, (n,), generator=g).cuda()
    huge, sign = torch.finfo(torch.float32).max, lambda n: (torch.randint(0, 2, (n,), generator=g) * 2 - 1).float().cuda()
    rows, columns = torch.arange(M, device="cuda"), torch.arange(N, device="cuda")
    if what == "rows of NaN":
        x[:] = NAN
    elif what == "a NaN a row":
        x[rows, at(M)] = NAN
    elif what == "an infinity a row":
        x[rows, at(M)] = INF * sign(M)
    elif what == "a NaN a column":
        w[columns, at(N)] = NAN
    elif what == "an infinity a column":
        w[columns, at(N)] = INF * sign(N)
    elif what == "a huge weight a column":
        x.mul_(2.0 ** -20)
        w[columns, at(N)] = huge * sign(N)
    else:      # some of each, and clean rows and columns between them
        x.mul_(2.0 ** -20)
        for k, v in enumerate((NAN, INF, -INF, huge, -huge, 0.0)):
            x[17 * k + 3::101, 5 * k + 2] = v
            w[29 * k + 1::97, 7 * k + 4] = v
    return x, w


SPRINKLED = ["rows of NaN", "a NaN a row", "an infinity a row", "a NaN a column", "an infinity a column", "a huge weight a column", "some of each"]


@pytest.mark.gpu
@pytest.mark.parametrize("what", SPRINKLED)
@pytest.mark.parametrize("tile,M,N,K", [((128, 256), 150, 528, 1024), ((64, 128), 300, 400, 384)])
def test_sums_that_are_no_numbers(what, tile, M, N, K):
    """NaN and infinities where a sum of float products has them, and numbers within their bound everywhere else."""
    from burn_lm_amd.csrc import ops
    x, w = sprinkled(M, N, K, what)
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    got = ops.gemm_split(ops.split_rows(x), w, torch.empty(M, N, device="cuda"), tile=tile)
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isposinf(), want.float().isposinf()) and torch.equal(got.isneginf(), want.float().isneginf())
    fine = want.isfinite() & (size < 1e38)
    assert bool(((got.double() - want).abs()[fine] <= (K + 2) * 2.0 ** -24 * size[fine]).all())


@pytest.mark.gpu
@pytest.mark.parametrize("what", SPRINKLED)
def test_sums_that_are_no_numbers_in_time(what):
    """Such a product stays within a few times a clean one's time (where every sum was walked one lane at a time: some hundred times)."""
    from burn_lm_amd.csrc import ops
    M, N, K = 512, 2048, 2048

    def us(x, w):
        parts, out, times = ops.split_rows(x), torch.empty(M, N, device="cuda"), []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            ops.gemm_split(parts, w, out, tile=(128, 256))
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 1e3)
        return sorted(times)[2]

    clean, these = us(*operands(M, N, K)), us(*sprinkled(M, N, K, what))
    print(f"{what}: {these:.0f} us, clean {clean:.0f}")
    assert these < 16 * clean


@pytest.mark.gpu
@pytest.mark.parametrize("M", [200, 700])
@pytest.mark.parametrize("K", [256, 2048, 2052, 4096])
def test_runtime_takes_every_form(M, K, monkeypatch):
    """linear and gated_linear where the parts are the faster way: bound weights and plain ones, planes, given tensors (also ones whose
    rows start where the parts' kernel does not store), rows with a stride, widths that have no parts."""
    from burn_lm_amd.csrc import ops
    from burn_lm_amd.engine.runtime import Runtime
    seen = []
    split = ops.gemm_split
    monkeypatch.setattr(ops, "gemm_split", lambda *a, **k: seen.append(a[1].shape) or split(*a, **k))
    rt = Runtime(torch.float32, "cuda:0")
    x, w = operands(M, 2048, K, pad=8)
    for weight in (rt.weight(w), w):
        check(rt.linear(x, weight), x, w)
        got = rt.linear(x, weight, partials=True)
        check(got.sum(0) if got.dim() == 3 else got, x, w)
        for room in (4, 3):
            given = torch.full((M, 2048 + room), NAN, device="cuda")
            check(rt.linear(x, weight, out=given[:, :2048]), x, w)
            assert bool(given[:, 2048:].isnan().all())
    check(rt.gated_linear(x, rt.weight(w, gated=True)), x, w, gated=True)
    check(rt.gated_linear(x, w), x, w, gated=True)
    if K == 2052 or (M, K) == (700, 2048):
        assert bool(seen) == (K == 2048)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [17, 40, 100])
@pytest.mark.parametrize("N,K", [(3072, 2048), (330, 2052), (528, 1152)])
def test_whole_results_of_planes(M, N, K, monkeypatch):
    """Few rows of few columns that have to come whole run in groups of K whose planes a pass adds: new tensors and given ones; where
    rows do not lie one behind the other the product writes them itself."""
    from burn_lm_amd.csrc import ops
    from burn_lm_amd.engine.runtime import Runtime
    added = []
    planes = ops.sum_planes
    monkeypatch.setattr(ops, "sum_planes", lambda y, out: added.append(y.shape[0]) or planes(y, out))
    rt = Runtime(torch.float32, "cuda:0")
    x, w = operands(M, N, K, pad=4)
    whole = rt.linear(x, w)
    assert whole.shape == (M, N) and added
    check(whole, x, w)
    given = torch.full((M, N), NAN, device="cuda")
    assert rt.linear(x, w, out=given) is given and torch.equal(given, whole)
    added.clear()
    wide = torch.full((M, N + 4), NAN, device="cuda")
    check(rt.linear(x, w, out=wide[:, :N]), x, w)
    assert not added and bool(wide[:, N:].isnan().all())


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,K,nh,nkv,hd", [(17, 128, 2, 1, 64), (130, 256, 3, 1, 48), (64, 384, 5, 1, 36 * 4), (100, 128, 2, 2, 20 * 4), (300, 256, 8, 4, 4)])
def test_projection_with_rotation_and_pages(tile, M, K, nh, nkv, hd):
    """Queries and pages are those of the same product followed by the rotation kernel (a rotation is two products and a sum: an ulp of the larger
    one apart at most), also of what is no finite number; rows of no sequence write no page, heads may end inside a tile of columns."""
    from burn_lm_amd.csrc import ops
    g = torch.Generator().manual_seed(M + K)
    N, page = (nh + 2 * nkv) * hd, 64
    x, w = operands(M, N, K)
    w.mul_(K ** -0.5)
    x[M - 1, 3], w[nh * hd + 1, 9], x[5, 9] = INF, NAN, 0.0
    pos = ((torch.arange(M) * 37 + 5) % 250).int().cuda()
    seq = torch.arange(M, dtype=torch.int32)
    seq[1] = -1
    seq, table = seq.cuda(), torch.randperm(4 * M, generator=g).view(M, 4).int().cuda()
    cs = torch.randn(256, hd // 2, 2, generator=g).cuda()
    got = []
    for fused in (True, False):
        k, v = (torch.full((4 * M, nkv, *s), 9.0, device="cuda") for s in ((page, hd), (hd, page)))
        for store in (False, True):
            out = torch.full((M, N), 7.0, device="cuda")
            if fused:
                ops.gemm_split_qkv_rope(x, w, out, pos, seq, table, cs, k, v, page, nh, nkv, hd, write_kv=store, tile=tile)
                assert bool((out[:, nh * hd:] == 7).all())
            else:
                ops.gemm_split(ops.split_rows(x), w, out, tile=tile)
                ops.rope_kv_write(out, pos, seq, table, cs, k, v, page, nh, nkv, hd, 0, write_kv=store)
            assert store or bool((k == 9).all() and (v == 9).all())
        got.append((out[:, :nh * hd][seq >= 0], k, v))
    for a, b in zip(*got):
        assert torch.allclose(a, b, rtol=2.0 ** -21, atol=2.0 ** -20, equal_nan=True)


@pytest.mark.gpu
def test_refused():
    from burn_lm_amd.csrc import ops
    x, w = operands(40, 64, 256)
    parts, out = ops.split_rows(x), torch.empty(40, 64, device="cuda")
    for bad in (lambda: ops.split_rows(x[:, :250]), lambda: ops.split_rows(x[:, 1:]), lambda: ops.split_rows(x.bfloat16()),
                lambda: ops.gemm_split(parts, w[:63], out[:, :63]), lambda: ops.gemm_split(parts[:2], w, out), lambda: ops.gemm_split(parts, w, out, tile=(64, 64)),
                lambda: ops.gemm_split(parts, w, torch.empty(3, 40, 64, device="cuda")), lambda: ops.gemm_split(parts, w[:, :200].contiguous(), out),
                lambda: ops.gemm_split(parts, w, out[:, :32], gated=True, tile=(128, 128)), lambda: ops.gemm_split(parts, w.half(), out)):
        with pytest.raises(ops.KernelError):
            bad()


def test_plan_keeps_its_bounds():
    """Sizes that the kernel does not have get no plan; groups of K are whole, and none is empty."""
    from burn_lm_amd.engine.runtime import split_plan
    for K in (4, 130, 2052):
        assert split_plan(100, 64, K, 256) is None
    assert split_plan(100, 60, 256, 256) is None
    # lanes' offsets into the weights are 32 bits: 256 columns of 2^22, and of the gated product all gate columns besides
    assert split_plan(100, 16, 1 << 22, 256) is None and split_plan(100, 16, (1 << 22) - 128, 256) is not None
    assert split_plan(100, 1 << 19, 2048, 256, gated=True) is None and split_plan(100, 1 << 19, 2048, 256) is not None
    for M in (17, 65, 1000):
        for N in (16, 2048, 5008):
            for K in (128, 1152, 2176, 4224, 8192):
                tile, groups, us = split_plan(M, N, K, 256, planes=True)
                assert tile in TILES and (groups - 1) * -(-K // 128 // groups) * 128 < K
                tile, groups, _ = split_plan(M, N, K, 256, added=True)
                assert tile in TILES and (groups - 1) * -(-K // 128 // groups) * 128 < K
                assert split_plan(M, N, K, 256)[1] == 1 and split_plan(M, N, K, 256, gated=True)[0][1] == 256 and us > 0
