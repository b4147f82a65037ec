"""The float32 attention on the matrix cores against 64 bits and against the generic kernel: prompts in portions, single tokens,
head sizes that are no multiples of sixteen, groups that fill no block or more than one, windows, cut key ranges.

The bound: a score of a query and a key is off by at most (head_dim + 3) 2^-24 times the sum of its products' sizes (times the
scale), a probability by twice the largest of these (its own and the maximum's), and the sums over n keys by (n + 8) 2^-24,
each against the largest value that the query sees."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
EPS, PAGE = 2.0 ** -24, 64


def case(lens, nkv, hd, seed, spare=3):
    """Pages in scrambled order whose unused places hold NaN -> (table, keys, values per sequence, key pages, value pages)."""
    g = torch.Generator().manual_seed(seed)
    need = [-(-n // PAGE) for n in lens]
    order = torch.randperm(sum(need) + spare, generator=g).tolist()
    table = torch.zeros(len(lens), max(need) + 1, dtype=torch.int32)
    kc, vc = torch.full((len(order), nkv, PAGE, hd), float("nan")), torch.full((len(order), nkv, hd, PAGE), float("nan"))
    keys, values = [], []
    for b, n in enumerate(lens):
        k, v = torch.randn(n, nkv, hd, generator=g), torch.randn(n, nkv, hd, generator=g)
        keys.append(k); values.append(v)
        for p in range(need[b]):
            page = table[b, p] = order.pop()
            part = slice(p * PAGE, min(n, (p + 1) * PAGE))
            kc[page, :, : part.stop - part.start] = k[part].transpose(0, 1)
            vc[page, :, :, : part.stop - part.start] = v[part].permute(1, 2, 0)
    return table, keys, values, kc, vc


def check(got, q, k, v, pos, scale, window, group):
    """got, q [heads, hd] at position pos over its sequence's keys and values [n, groups, hd]."""
    lo = max(0, pos - window + 1) if window else 0
    k, v = (t[lo: pos + 1].double().repeat_interleave(group, 1) for t in (k, v))
    q = q.double()
    want = torch.einsum("hn,nhd->hd", torch.softmax(torch.einsum("hd,nhd->hn", q, k) * scale, -1), v)
    off = (q.shape[1] + 3) * EPS * scale * torch.einsum("hd,nhd->hn", q.abs(), k.abs()).amax(1)
    bound = (2 * off + (k.shape[0] + 8) * EPS) * v.abs().amax((0, 2))
    assert bool(((got.double() - want).abs() <= bound[:, None]).all()), float(((got.double() - want).abs() / bound[:, None]).max())


SHAPES = [(4, 4, 64), (8, 2, 64), (6, 1, 24), (5, 1, 4), (40, 2, 16), (6, 2, 128), (8, 1, 100), (3, 3, 72), (7, 1, 96), (6, 2, 36), (4, 2, 48), (5, 1, 60)]


@pytest.mark.parametrize("window", [0, 1, 70])
@pytest.mark.parametrize("nh,nkv,hd", SHAPES)
def test_prompts(nh, nkv, hd, window):
    from burn_lm_amd.csrc import ops
    lens, new = [150, 333, 65, 1, 40, 64], [150, 70, 1, 1, 33, 64]
    table, keys, values, kc, vc = case(lens, nkv, hd, 3)
    positions = [p for n, m in zip(lens, new) for p in range(n - m, n)]
    cu = [sum(new[:b]) for b in range(len(new) + 1)]
    stride = -(-((nh + 2 * nkv) * hd) // 8) * 8
    qkv = torch.randn(cu[-1] + 2, stride, generator=torch.Generator().manual_seed(4))       # two rows of no sequence behind them
    out = torch.full((cu[-1] + 2, nh * hd), 7.0, device="cuda")
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    args = (i32(positions + [0, 0]),)
    assert ops.attn_f32_supported(qkv.cuda(), stride, kc.cuda(), vc.cuda(), hd, PAGE)
    ops.attn_prefill_f32(qkv.cuda(), stride, out, *args, i32(cu), table.cuda(), kc.cuda(), vc.cuda(), PAGE, len(lens), max(new), nh, nkv, hd,
                         hd ** -0.5, window)
    got = out.cpu().reshape(-1, nh, hd)
    assert bool((got[cu[-1]:] == 7.0).all())
    for b in range(len(lens)):
        for t in range(cu[b], cu[b + 1], 1 if new[b] < 50 else 7):
            check(got[t], qkv[t, : nh * hd].reshape(nh, hd), keys[b], values[b], positions[t], hd ** -0.5, window, nh // nkv)


@pytest.mark.parametrize("lens,nh,nkv", [([600], 8, 1), ([520, 30, 1100], 12, 3), ([1040], 4, 4)])
def test_prompts_of_many_places(lens, nh, nkv):
    """More than 32 blocks a key-value head: whole runs of 32 that go the other way round, and runs that are cut short."""
    from burn_lm_amd.csrc import ops
    hd, group = 16, nh // nkv
    table, keys, values, kc, vc = case(lens, nkv, hd, 5)
    cu = [sum(lens[:b]) for b in range(len(lens) + 1)]
    qkv = torch.randn(cu[-1], (nh + 2 * nkv) * hd, generator=torch.Generator().manual_seed(6))
    out = torch.full((cu[-1], nh * hd), 7.0, device="cuda")
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    ops.attn_prefill_f32(qkv.cuda(), qkv.shape[1], out, i32([p for n in lens for p in range(n)]), i32(cu), table.cuda(), kc.cuda(), vc.cuda(), PAGE,
                         len(lens), max(lens), nh, nkv, hd, hd ** -0.5, 0)
    got = out.cpu().reshape(-1, nh, hd)
    for b, n in enumerate(lens):
        for t in list(range(0, n, 61)) + [n - 1]:
            check(got[cu[b] + t], qkv[cu[b] + t, : nh * hd].reshape(nh, hd), keys[b], values[b], t, hd ** -0.5, 0, group)


@pytest.mark.parametrize("hd", [4, 64])
def test_prompts_probabilities(hd):
    """Every query sees one key with score zero, one with a score of its own and others that are out of sight, and the value of the second alone is one:
    the result is the exponential, and an ulp is what the library promises for it, also where that is below 2^-126."""
    from burn_lm_amd.csrc import ops
    nh, n = 64, 64
    g = torch.Generator().manual_seed(hd)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    q, keys, values = torch.zeros(n, (nh + 2) * hd), torch.zeros(PAGE, hd), torch.zeros(hd, PAGE)
    score = -17.0 - 86.0 * torch.rand(n, nh, generator=g)
    rows = q[:, : nh * hd].view(n, nh, hd)
    rows[..., 0], rows[..., 1] = score, 1.0
    keys[1, 0], keys[2:, 1], values[:, 1] = 1.0, -1e30, 1.0
    out = torch.empty(n, nh * hd, device="cuda")
    ops.attn_prefill_f32(q.cuda(), q.shape[1], out, i32(list(range(n))), i32([0, n]), i32([[0]]), keys[None, None].cuda(), values[None, None].cuda(), PAGE,
                         1, n, nh, 1, hd, 1.0, 0)
    got, want = out.cpu().view(n, nh, hd)[2:].double(), score[2:, :, None].double().exp()
    ulp = torch.exp2(torch.floor(torch.log2(want)).clamp_min(-126.0) - 23)
    assert bool(((got - want).abs() <= ulp).all()), float(((got - want).abs() / ulp).max())


@pytest.mark.parametrize("splits", [1, 2, 5])
@pytest.mark.parametrize("window", [0, 1, 70])
@pytest.mark.parametrize("nh,nkv,hd", SHAPES)
def test_single_tokens(nh, nkv, hd, window, splits):
    from burn_lm_amd.csrc import ops
    lens = [1, 64, 65, 333, 700]
    table, keys, values, kc, vc = case(lens, nkv, hd, 5)
    stride = -(-((nh + 2 * nkv) * hd) // 8) * 8
    qkv = torch.randn(len(lens) + 1, stride, generator=torch.Generator().manual_seed(6))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    for _ in range(2):         # the second call finds the counters as the first left them
        out = torch.full((len(lens) + 1, nh * hd), 7.0, device="cuda")
        ops.attn_decode_f32(qkv.cuda(), stride, out, i32([n - 1 for n in lens] + [0]), i32([0, 1, 2, 3, 4, -1]), table.cuda(), kc.cuda(), vc.cuda(),
                            PAGE, nh, nkv, hd, hd ** -0.5, window, splits)
        got = out.cpu().reshape(-1, nh, hd)
        assert bool((got[-1] == 0).all())       # a row of no sequence
        for b, n in enumerate(lens):
            check(got[b], qkv[b, : nh * hd].reshape(nh, hd), keys[b], values[b], n - 1, hd ** -0.5, window, nh // nkv)


@pytest.mark.parametrize("window", [0, 100])
@pytest.mark.parametrize("nh,nkv,hd", [(8, 2, 64), (3, 1, 128), (4, 4, 20)])
@pytest.mark.parametrize("pages", [1, 2, 3, 4, 5, 8, 9, 10, 11, 12, 13])
def test_last_rounds_in_halves_and_quarters(nh, nkv, hd, pages, window):
    """Rounds of the eight wavefronts with whole pages, and a last one in halves or quarters of pages, the last key in each of them."""
    from burn_lm_amd.csrc import ops
    lens = [pages * PAGE - less for less in (63, 48, 33, 32, 17, 1, 0)]
    table, keys, values, kc, vc = case(lens, nkv, hd, pages)
    q = torch.randn(len(lens), nh * hd, generator=torch.Generator().manual_seed(6))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    out = torch.full((len(lens), nh * hd), 7.0, device="cuda")
    ops.attn_decode_f32(q.cuda(), nh * hd, out, i32([n - 1 for n in lens]), i32(range(len(lens))), table.cuda(), kc.cuda(), vc.cuda(), PAGE, nh, nkv, hd,
                        hd ** -0.5, window, 1)
    for b, n in enumerate(lens):
        check(out[b].cpu().reshape(nh, hd), q[b].reshape(nh, hd), keys[b], values[b], n - 1, hd ** -0.5, window, nh // nkv)


@pytest.mark.parametrize("bad", [math.inf, -math.inf, math.nan])
def test_values_that_are_no_numbers_stay_with_those_that_see_them(bad):
    """A token whose value (or key) is infinite or no number: earlier queries and queries whose window has passed it agree with
    the generic kernel, in prompts and for single tokens, and so do the others, number by number."""
    from burn_lm_amd.csrc import ops
    nh, nkv, hd, n, window = 4, 2, 64, 150, 40
    stride = (nh + 2 * nkv) * hd
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    qkv = torch.randn(n, stride, generator=torch.Generator().manual_seed(8)).cuda()
    for what in ("value", "key"):
        table, keys, values, kc, vc = case([n], nkv, hd, 7)
        page = table[0, 1]
        if what == "value":
            vc[page, 1, 5, 70 - 64] = bad
        else:
            kc[page, 1, 70 - 64, 5] = bad
        table, kc, vc = table.cuda(), kc.cuda(), vc.cuda()
        want, got = (torch.full((n, nh * hd), 7.0, device="cuda") for _ in range(2))
        ops.attn_paged_init()
        ops.attn_paged(qkv, stride, want, i32(range(n)), i32([0] * n), table, kc, vc, PAGE, nh, nkv, hd, 0.125, window, 1)
        ops.attn_prefill_f32(qkv, stride, got, i32(range(n)), i32([0, n]), table, kc, vc, PAGE, 1, n, nh, nkv, hd, 0.125, window)
        for t in (got, ):
            assert torch.equal(t.isnan(), want.isnan()) and torch.equal(t.isinf(), want.isinf())
            fine = want.isfinite()
            assert float((t - want)[fine].abs().max()) < 1e-5       # two sums of at most 40 values below 5, in other orders
        for pos in (60, 70, 100, 109, 110, 149):
            one = torch.empty(1, nh * hd, device="cuda")
            ops.attn_decode_f32(qkv[pos: pos + 1], stride, one, i32([pos]), i32([0]), table, kc, vc, PAGE, nh, nkv, hd, 0.125, window, 1)
            assert torch.equal(one[0].isnan(), want[pos].isnan()) and torch.equal(one[0].isinf(), want[pos].isinf()), pos


def test_refused():
    from burn_lm_amd.csrc import ops
    z, out = torch.zeros(2, 24, device="cuda"), torch.zeros(2, 8, device="cuda")
    i = torch.zeros(2, dtype=torch.int32, device="cuda")
    for hd, page in ((6, 64), (132, 64), (64, 32)):
        kc, vc = torch.zeros(1, 1, page, hd, device="cuda"), torch.zeros(1, 1, hd, page, device="cuda")
        assert not ops.attn_f32_supported(z, 24, kc, vc, hd, page)
    kc, vc = torch.zeros(1, 1, 64, 8, device="cuda"), torch.zeros(1, 1, 8, 64, device="cuda")
    with pytest.raises(ops.KernelError):
        ops.attn_decode_f32(z[:, 1:], 24, out, i, i, i.view(2, 1), kc, vc, 64, 1, 1, 8, 1.0)
    with pytest.raises(ops.KernelError):
        ops.attn_prefill_f32(z, 22, out, i, i[:2], i.view(2, 1), kc, vc, 64, 1, 1, 1, 1, 8, 1.0)
