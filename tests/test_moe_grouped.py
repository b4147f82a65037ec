"""Experts of many rows: every token through its own experts only, against 64 bits and against all through all.

The bound: a token's gated activations are rounded to bfloat16 once (2^-9 of their size each) and all sums are float32, so a
result is off by at most 2^-9 times the sum of its products' sizes, and as much again for the float32 sums of up to 2,048."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -8


def choices(T, E, top, g, kind):
    w = torch.zeros(T, E + 1)
    if kind == "one":                                    # every token the same experts: the others have no rows
        idx = torch.arange(top).expand(T, top)
    else:
        idx = torch.rand(T, E, generator=g).argsort(1)[:, :top]
    w.scatter_(1, idx, torch.rand(T, top, generator=g) + 0.1)
    if kind == "missing":                                # tokens with fewer experts, or none
        w[:, :E][torch.rand(T, E, generator=g) < 0.4] = 0
        w[T // 2] = 0
    w[:, E] = 7.0
    return w


@pytest.mark.parametrize("kind", ["all", "one", "missing"])
@pytest.mark.parametrize("T,E,top,f,D", [(1, 2, 1, 64, 64), (130, 3, 2, 64, 192), (257, 16, 4, 192, 128), (1100, 5, 5, 128, 320),
                                         (300, 128, 8, 64, 64)])
def test_kernels(T, E, top, f, D, kind):
    from burn_lm_amd.csrc import ops
    g = torch.Generator().manual_seed(T + E)
    x, gu, down = (torch.randn(*s, generator=g).mul_(s[1] ** -0.5 if s[0] != T else 1).bfloat16()
                   for s in ((T, D), (2 * E * f, D), (D, E * f)))
    w = choices(T, E, top, g, kind)
    y = ops.moe_grouped(x.cuda(), gu.cuda(), down.cuda(), w.cuda(), E, top)
    assert y.shape == (top, T, D)
    both = x.double() @ gu.double().t()
    act = torch.nn.functional.silu(both[:, :E * f]) * both[:, E * f:] * w[:, :E].double().repeat_interleave(f, 1)
    want, bound = act @ down.double().t(), EPS * (act.abs() @ down.double().abs().t()) + 1e-6
    assert ((y.double().sum(0).cpu() - want).abs() <= bound).all()
    # a token's result does not depend on the others, nor on their number
    rows = torch.randperm(T, generator=g)[: T // 2 + 1]
    again = ops.moe_grouped(x[rows].cuda(), gu.cuda(), down.cuda(), w[rows].contiguous().cuda(), E, top)
    assert torch.equal(again, y[:, rows.cuda()])


@pytest.mark.parametrize("T,E,top,f,D", [(130, 3, 2, 64, 192), (900, 16, 4, 128, 256), (70, 128, 8, 64, 64)])
def test_a_table_of_the_tokens(T, E, top, f, D):
    """The same bits as with the table's weights made first; ids outside the table, ids that wait on the device, entries that repeat."""
    from burn_lm_amd.csrc import ops
    g = torch.Generator().manual_seed(T)
    V = 40
    x, gu, down = (torch.randn(*s, generator=g).bfloat16().cuda() for s in ((T, D), (2 * E * f, D), (D, E * f)))
    table = torch.rand(V, E, generator=g).argsort(1)[:, :top].int()
    table[3, 1] = table[3, 0]
    table, ids = table.cuda(), torch.randint(0, V, (T,), generator=g).int()
    ids[5], ids[9], ids[7] = V, -1, 3
    ids = ids.cuda()
    picked, rows = torch.randint(0, V, (64,), generator=g).int().cuda(), torch.full((T,), -1, dtype=torch.int32)
    rows[::3] = 7
    source = rows.cuda(), torch.tensor([picked.data_ptr()], dtype=torch.int64, device="cuda")
    for source in (None, source):
        weights = torch.empty(T, E + 1, device="cuda")
        ops.moe_table(table, ids, weights, E, source)
        want = ops.moe_grouped(x, gu, down, weights, E, top)
        assert torch.equal(ops.moe_grouped(x, gu, down, None, E, top, table=table, ids=ids, token_source=source), want)


def part_tiles(rows, n_tiles, units):
    """What moe_duo_kernel runs behind its whole tiles for these rows of the experts (K >= 1,024): 1: an expert's last rows as a half, 2:
    halves only, 3: tiles of 160 rows only."""
    up = lambda a, b: -(-a // b)
    wholes, lone = sum(r // 256 + (r % 256 > 128) for r in rows) * n_tiles, sum(0 < r % 256 <= 128 for r in rows) * n_tiles
    rest = wholes % units
    mixed = wholes // units * 100 + (100 if rest else 0) + up(max(0, lone - (units - rest if rest else 0)), units) * 57
    halves, fives = (up(sum(up(r, size) for r in rows) * n_tiles, units) * cost for size, cost in ((128, 57), (160, 71)))
    return 3 if fives < min(halves, mixed) else 2 if halves < mixed else 1


@pytest.mark.parametrize("rows", [[500, 530, 640, 641], [160, 161, 0, 1], [1000, 20, 300, 700], [320, 321, 160, 159]])
def test_tiles_of_five_eighths(rows):
    """Experts whose rows end at, behind and in front of tiles of 160 rows, alone on a few units: halves, wholes and five eighths (which
    the number of units decides) give the same bits, and those of the small tiles."""
    from burn_lm_amd.csrc import ops
    E, f, D = 4, 1024, 1024
    T = sum(rows)
    all_units = (8, 11, 16, 17, 36, 40, 64, 70, 80, 96, 112, 128, 150, 256, 2000)
    about = (T + 64 * E) // 128
    for n_tiles, most in ((f // 128, about * (f // 128) * 5 // 2), (D // 256, about * (D // 256))):      # both products reach them
        assert any(part_tiles(rows, n_tiles, u) == 3 for u in all_units if u <= most)
    g = torch.Generator().manual_seed(T)
    x, gu, down = (torch.randn(*s, generator=g).mul_(s[1] ** -0.5).bfloat16().cuda() for s in ((T, D), (2 * E * f, D), (D, E * f)))
    w = torch.zeros(T, E + 1)
    w[torch.arange(T), torch.repeat_interleave(torch.arange(E), torch.tensor(rows))[torch.randperm(T, generator=g)]] = 0.5
    w, lists, act = w.cuda(), torch.empty(2 * E * T + E, dtype=torch.int32, device="cuda"), torch.empty(T, f, dtype=torch.bfloat16, device="cuda")
    results = []
    for units in all_units:
        planes = torch.full((1, T, D), float("nan"), device="cuda")
        ops._call("blm_moe_grouped", x.data_ptr(), D, gu.data_ptr(), down.data_ptr(), w.data_ptr(), E + 1, None, None, None, None, 0,
                  planes.data_ptr(), lists.data_ptr(), lists.data_ptr() + 8 * E * T, act.data_ptr(), T, D, E, f, 1, units, ops._stream())
        results.append(planes)
    assert not results[0].isnan().any() and all(torch.equal(r, results[0]) for r in results[1:])


def test_weights_that_are_no_numbers():
    from burn_lm_amd.csrc import ops
    T, E, top, f, D = 150, 4, 2, 64, 64
    g = torch.Generator().manual_seed(0)
    x, gu, down = (torch.randn(*s, generator=g).bfloat16().cuda() for s in ((T, D), (2 * E * f, D), (D, E * f)))
    w = choices(T, E, top, g, "all")
    plain = ops.moe_grouped(x, gu, down, w.cuda(), E, top)
    w[5] = float("nan")
    y = ops.moe_grouped(x, gu, down, w.cuda(), E, top)
    others = torch.arange(T) != 5
    assert y[:, 5].isnan().all() and torch.equal(y[:, others.cuda()], plain[:, others.cuda()])


def test_refusals():
    from burn_lm_amd.csrc import ops
    from burn_lm_amd.csrc.ops import KernelError
    x, gu, down, w = (torch.zeros(*s, dtype=torch.bfloat16, device="cuda") for s in ((4, 64), (256, 64), (64, 128), (4, 3)))
    for bad in (dict(x=x.float()), dict(gu=gu[:128]), dict(down=down[:32]), dict(weights=w), dict(top=3), dict(x=x[:, :32].contiguous())):
        a = dict(x=x, gu=gu, down=down, weights=w.float(), top=2) | bad
        with pytest.raises(KernelError):
            ops.moe_grouped(a["x"], a["gu"], a["down"], a["weights"], 2, a["top"])


@pytest.mark.parametrize("kind", ["router", "groups", "table"])
def test_parts_take_either_way(kind, monkeypatch):
    """A step of many rows through the parts, against the same step with every expert for every token: that form rounds gates,
    ups and activations to bfloat16 (three times 2^-9), this one the activations once."""
    import burn_lm_amd.parts.routed_experts as RE
    from burn_lm_amd.engine.runtime import Runtime
    rt, g = Runtime(), torch.Generator().manual_seed(3)
    T, D, E, top, f = 700, 128, 8, 2, 64
    names = {n: n for n in ["router", "router_bias", "correction", "table"] + [f"e{e}.{r}" for e in range(E) for r in ("gate", "up", "down")]}
    n_router = E + 2 if kind == "groups" else E
    t = {f"e{e}.{r}": (torch.randn(*((D, f) if r == "down" else (f, D)), generator=g) * D ** -0.5).bfloat16().cuda()
         for e in range(E) for r in ("gate", "up", "down")}
    t["router"] = torch.randn(n_router, D, generator=g).bfloat16().cuda()
    t["router_bias"], t["correction"] = torch.randn(E, generator=g).cuda(), torch.randn(n_router, generator=g).cuda()
    t["table"] = torch.rand(50, E, generator=g).argsort(1)[:, :top].int().cuda()
    params = dict(width=D, experts=E, top=top, expert_inner=f, vocab=50, identity=2)
    part = dict(router=RE.RoutedExperts, groups=RE.GroupedRoutedExperts, table=RE.TableExperts)[kind](params, names)
    part.bind(t, rt)

    class Step:
        token_ids = torch.randint(-1, 50, (T,), generator=g).int().cuda()     # -1: a row of no token
        token_source = None
    x = torch.randn(T, D, generator=g).bfloat16().cuda()
    add = lambda terms: sum((y.y.double().sum(0) if y.y.dim() == 3 else y.y.double()) * (1 if y.row is None else y.row.double()[:, None]) for y in terms)
    assert part._grouped(T)
    terms = part.forward_terms(x, Step)
    assert terms[0].y.shape == (top, T, D)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        recorded = part.forward_terms(x, Step)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded[0].y, terms[0].y)
    monkeypatch.setattr(RE, "GROUPED_MIN_ROWS", T + 1)
    assert not part._grouped(T)
    want, got = add(part.forward_terms(x, Step)), add(terms)
    assert (got - want).norm() <= 3 * 2 ** -9 * want.norm()
    if kind == "table":
        assert got[Step.token_ids < 0].abs().max() == 0


@pytest.mark.parametrize("form", ["columns of wider rows", "odd address"])
def test_rows_that_the_grouped_form_does_not_take(form):
    """Rows with a stride or at an address of their own go through all experts: the part takes what it always took."""
    import burn_lm_amd.parts.routed_experts as RE
    from burn_lm_amd.engine.runtime import Runtime
    rt, g = Runtime(), torch.Generator().manual_seed(3)
    T, D, E, top, f = 700, 128, 8, 2, 64
    t = {f"e{e}.{r}": (torch.randn(*((D, f) if r == "down" else (f, D)), generator=g) * D ** -0.5).bfloat16().cuda()
         for e in range(E) for r in ("gate", "up", "down")}
    t["router"], t["router_bias"] = torch.randn(E, D, generator=g).bfloat16().cuda(), torch.zeros(E).cuda()
    part = RE.RoutedExperts(dict(width=D, experts=E, top=top, expert_inner=f), {n: n for n in t})
    part.bind(t, rt)
    x = torch.randn(T, D, generator=g).bfloat16().cuda()
    if form == "odd address":
        given = torch.empty(T * D + 8, dtype=x.dtype, device="cuda")[1:1 + T * D].view(T, D)
    else:
        given = torch.empty(T, D + 8, dtype=x.dtype, device="cuda")[:, :D]
    given.copy_(x)
    assert part._grouped(T)
    want, got = ((lambda y: y.double().sum(0) if y.dim() == 3 else y.double())(part.forward(v, None)) for v in (x, given))
    assert (got - want).norm() <= 3 * 2 ** -9 * want.norm()


def test_no_more_memory_than_the_stacked_form():
    """Many rows of a wide model with narrow experts: planes for every choice would take several times what all experts' activations
    take."""
    from types import SimpleNamespace as NS

    from burn_lm_amd.csrc import ops
    from burn_lm_amd.parts.routed_experts import RoutedExperts

    def grouped(rows, width, inner, experts, top):
        part = RoutedExperts.__new__(RoutedExperts)
        part.rt, part.E, part.top, part.f, part.s = NS(ops=ops, dtype=torch.bfloat16), experts, top, inner, 0
        matrix = lambda *shape: NS(w=torch.empty(shape, dtype=torch.bfloat16, device="meta"))
        part.w_gate_up, part.w_down = matrix(2 * experts * inner, width), matrix(width, experts * inner)
        return part._grouped(rows)
    assert grouped(2048, 4096, 64, 64, 8)                                    # 0.3 GB
    assert not grouped(131072, 4096, 64, 64, 8)                              # 17 GB against 3
    assert grouped(65536, 2048, 512, 16, 4) and grouped(65536, 1024, 128, 128, 8)     # less than the stacked form


@pytest.mark.parametrize("kind", ["all", "one", "missing"])
@pytest.mark.parametrize("T,E,top,f,D,units",
                         [(257, 3, 2, 256, 256, 4), (257, 3, 2, 256, 256, 5), (700, 5, 2, 384, 640, 8), (700, 5, 2, 384, 640, 32),
                          (1030, 2, 1, 256, 384, 8), (1030, 2, 1, 256, 384, 18), (300, 64, 4, 256, 256, 8), (300, 64, 4, 256, 256, 40),
                          (4000, 4, 3, 384, 768, 256), (2100, 16, 4, 256, 1024, 256)])
def test_tiles_of_256(monkeypatch, T, E, top, f, D, units, kind):
    """The tiles of 256x256: experts with whole tiles, a half behind them, or halves only (the fewer units, the more rounds there are to
    choose by), with no rows at all, and columns that end within a tile.  Each of these takes them for gate and up and for
    down: as many halves, an expert's last one half full, as the launch asks for.  The bound as above."""
    from burn_lm_amd.csrc import ops
    about = (T * top + 64 * E) // 128
    assert about * -(-f // 128) * 5 >= 2 * units and about * -(-D // 256) >= units
    monkeypatch.setattr(ops, "compute_units", lambda index: units)
    test_kernels(T, E, top, f, D, kind)


@pytest.mark.parametrize("T", [8000, 400])
def test_gating_is_float32(T):
    """Two million gates of -64 to -16 that float32 holds exactly (a b + c d of bfloat16, steps of 2^-18), ups and weights of one, an
    identity behind them: in the tiles of many rows and in those of few, an activation is the bfloat16 next to a float32 silu, whose
    exponential, sum and division are off by at most 2^-22 of it together (2^-23, 2^-24 and 2^-24); twice that either way."""
    from burn_lm_amd.csrc import ops
    g = torch.Generator().manual_seed(1)
    D, wrong = 256, 0
    steps = lambda n, at, step: at + torch.randint(0, 128, (n,), generator=g) * step
    for _ in range(8000 // T):
        x, gu = torch.zeros(T, D), torch.zeros(2 * D, D)
        x[:, 0], x[:, 1], x[:, 2] = steps(T, -32, 2.0 ** -3), steps(T, 2.0 ** -4, 2.0 ** -11), 1.0
        gu[:D, 0], gu[:D, 1], gu[D:, 2] = steps(D, 1, 2.0 ** -7), steps(D, 1, 2.0 ** -7), 1.0
        y = ops.moe_grouped(x.bfloat16().cuda(), gu.bfloat16().cuda(), torch.eye(D).bfloat16().cuda(), torch.ones(T, 2).cuda(), 1, 1)[0].cpu()
        want = torch.nn.functional.silu(x.double() @ gu[:D].double().T)
        a, b = ((want * (1 + e * 2.0 ** -21)).bfloat16().float() for e in (-1, 1))
        wrong += int(((y < torch.minimum(a, b)) | (y > torch.maximum(a, b))).sum())
    assert wrong == 0


@pytest.mark.parametrize("T,E,top,f,D", [(700, 64, 16, 64, 64), (200, 200, 33, 64, 64), (1300, 9, 9, 64, 64), (1300, 16, 8, 64, 64), (900, 16, 3, 64, 64)])
def test_a_table_of_many_experts_a_token(T, E, top, f, D, monkeypatch):
    """Rows of up to eight experts make the lists themselves, longer ones (which every expert would compare entry by entry for every token)
    are made weights first; the same bits, also with entries that name no expert."""
    from burn_lm_amd.csrc import ops
    g = torch.Generator().manual_seed(T + top)
    x, gu, down = (torch.randn(*s, generator=g).bfloat16().cuda() for s in ((T, D), (2 * E * f, D), (D, E * f)))
    table = torch.rand(50, E, generator=g).argsort(1)[:, :top].int()
    table[3, 1] = table[3, 0]
    table[4, 0], table[4, 2], table[5, 1] = -1, E, -2 ** 31
    table, ids = table.cuda(), torch.randint(0, 50, (T,), generator=g).int().cuda()
    weights = torch.empty(T, E + 1, device="cuda")
    ops.moe_table(table, ids, weights, E)
    want, calls, real = ops.moe_grouped(x, gu, down, weights, E, top), [], ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (calls.append(name), real(name, *a))[1])
    assert torch.equal(ops.moe_grouped(x, gu, down, None, E, top, table=table, ids=ids), want)
    assert calls == (["blm_moe_table"] if top > 8 else []) + ["blm_moe_grouped"]
