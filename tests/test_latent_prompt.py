"""Latent attention over prompts with expanded keys and values: the kernels alone against 64 bits, and the part's choice between
them and the absorbed form over prompts, portions, unequal batches and recorded steps.

The bound for the kernels: keys, values, probabilities and results are rounded to bfloat16 once (2^-9 of their size each); a
score is then off by 2^-9 times the scale times the sum of its products' sizes, a probability by twice the largest of these."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
EPS, PAGE = 2.0 ** -9, 64


@pytest.mark.parametrize("sink", [False, True])
@pytest.mark.parametrize("window", [0, 1, 100])
@pytest.mark.parametrize("D,DR,R,H", [(64, 32, 64, 3), (64, 64, 128, 8), (128, 32, 192, 2), (128, 64, 512, 16)])
def test_kernels(D, DR, R, H, window, sink):
    from burn_lm_amd.csrc import ops
    g = torch.Generator().manual_seed(D + DR + R)
    lens, new = [150, 333, 64, 1, 200], [150, 129, 64, 1, 33]
    need = [-(-n // PAGE) for n in lens]
    order = torch.randperm(sum(need) + 2, generator=g).tolist()
    table = torch.full((len(lens) + 1, max(need) + 2), -1, dtype=torch.int32)
    kc = torch.full((len(order), 1, PAGE, R + DR), float("nan")).bfloat16()
    rows = []
    for b, n in enumerate(lens):
        r = torch.randn(n, R + DR, generator=g).bfloat16()
        rows.append(r)
        first = max(0, n - new[b] - window + 1) // PAGE if window else 0
        for p in range(first, need[b]):         # pages that the window has passed are somebody else's
            page = table[b, p] = order.pop()
            part = r[p * PAGE: (p + 1) * PAGE]
            kc[page, 0, : len(part)] = part
    wk, wv = (torch.randn(H * D, R, generator=g) * R ** -0.5 for _ in range(2))
    wk, wv = wk.bfloat16(), wv.bfloat16()
    T = sum(new) + 3                                   # three rows of no sequence, and a sequence that brings none
    ld = -(-(H * (D + DR) + 5) // 8) * 8
    q = torch.randn(T, ld, generator=g).bfloat16()
    turned = torch.randn(T, H, DR, generator=g).bfloat16()
    cu = [sum(new[:b]) for b in range(len(new) + 1)] + [sum(new)]
    positions = [p for n, m in zip(lens, new) for p in range(n - m, n)] + [0] * 3
    sinks = torch.randn(H, generator=g) * 2 if sink else None
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")

    class step:
        n_tokens, n_seqs, max_new, max_len_after = T, len(lens) + 1, max(new), max(lens)
        cu_seqlens, lens_after = i32(cu), i32(lens + [0])
    step.positions = i32(positions)
    scale, out = (D + DR) ** -0.5, torch.full((T, H * D), 7.0, dtype=torch.bfloat16, device="cuda")
    assert ops.latent_prompt_supported(torch.bfloat16, R, D, DR, D) and not ops.latent_prompt_supported(torch.float32, R, D, DR, D)
    ops.latent_prompt(q.cuda()[:, : H * (D + DR)], turned.cuda(), out, kc.cuda(), wk.cuda(), wv.cuda(), step, table.cuda(), max(need) + 1, H, R, D,
                      DR, D, scale, window=window, sinks=None if sinks is None else sinks.cuda())
    got = out.cpu().double().reshape(T, H, D)
    assert bool((got[cu[-1]:] == 7.0).all())
    for b, n in enumerate(lens):
        lat, kr = rows[b][:, :R].double(), rows[b][:, R:].double()
        k = torch.cat(((lat @ wk.double().t()).reshape(n, H, D), kr[:, None].expand(n, H, DR)), -1)
        v = (lat @ wv.double().t()).reshape(n, H, D)
        for t in range(cu[b], cu[b + 1], 5):
            pos = positions[t]
            lo = max(0, pos - window + 1) if window else 0
            qt = torch.cat((q[t, : H * (D + DR)].double().reshape(H, D + DR)[:, :D], turned[t].double()), -1)
            s = torch.einsum("hd,nhd->hn", qt, k[lo: pos + 1]) * scale
            off = scale * EPS * torch.einsum("hd,nhd->hn", qt.abs(), k[lo: pos + 1].abs()).amax(1)
            p = torch.softmax(torch.cat((s, sinks[:, None].double()), 1) if sink else s, -1)[:, : s.shape[1]]
            want, most = torch.einsum("hn,nhd->hd", p, v[lo: pos + 1]), v[lo: pos + 1].abs().amax((0, 2))
            bound = (2 * off + 4 * EPS)[:, None] * most[:, None] + 1e-6
            assert bool(((got[t] - want).abs() <= bound).all()), (b, t, float(((got[t] - want).abs() / bound).max()))


@pytest.mark.parametrize("D,DR", [(64, 32), (64, 64), (128, 32), (128, 64)])
def test_probabilities_add_up_to_one(D, DR):
    """Every value is one, so every result is: the weights that meet the values and the denominator are the same numbers.  All
    keys but the first have a probability of just under half a rounding step above a half of the first's; a denominator of
    unrounded ones would come out 2^-8 too large."""
    from burn_lm_amd.csrc import ops
    R, T = 64, 200
    wk, wv = torch.zeros(D, R), torch.zeros(D, R)
    wk[0, 1] = wv[:, 0] = 1
    kc = torch.zeros(4, 1, PAGE, R + DR)
    kc.view(-1, R + DR)[:T, 0] = 1            # every row's value: ones
    kc.view(-1, R + DR)[0, 1] = 1             # the first row's key
    q = torch.zeros(T, D + DR)
    q[:, 0] = 1
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    b16 = lambda x: x.bfloat16().cuda()

    class step:
        n_tokens, n_seqs, max_new, max_len_after = T, 1, T, T
        cu_seqlens, lens_after, positions = i32([0, T]), i32([T]), i32(list(range(T)))
    out = torch.zeros(T, D, dtype=torch.bfloat16, device="cuda")
    scale = -math.log(0.5 + 0.97 * EPS)
    ops.latent_prompt(b16(q), torch.zeros(T, 1, DR, dtype=torch.bfloat16, device="cuda"), out, b16(kc), b16(wk), b16(wv), step, i32([[0, 1, 2, 3]]), 4, 1,
                      R, D, DR, D, scale)
    assert bool((out == 1).all()), float(out.min())


def small_netanex(window):
    """One layer of differential, latent and gated attention each, sizes that the expanded form takes."""
    moe = dict(kind="moe", expert=dict(ff=32), router=dict(experts=4, top=2))
    latent = dict(heads=4, dim=64, rot_dim=32, vdim=64, kv_rank=128, scale=96 ** -0.5, rot=dict(base=10000.0, dims=32))
    if window:
        latent["mask"] = dict(size=window)
    layers = [dict(type="latent_attention", mlp=moe, mixer=dict(latent)), dict(type="latent_attention", mlp=moe, mixer=dict(latent))]
    return dict(architecture="Netanex", vocab=97, width=128, norm=dict(eps=1e-6), layers=layers)


@pytest.mark.parametrize("window", [0, 80])
def test_the_part_takes_either_form(window, monkeypatch):
    """The same schedule with and without the expanded form: whole prompts, portions behind others, unequal batches, single tokens
    behind them, the same shapes again from recorded steps.  bfloat16 roundings of two forms of the same sums: 2 % of the largest
    logit over two layers."""
    import burn_lm_amd.parts.latent_attention as part
    from burn_lm_amd.csrc import ops
    from burn_lm_amd.engine.loading import random_engine
    calls = []
    real = ops.latent_prompt
    monkeypatch.setattr(ops, "latent_prompt", lambda *a, **k: calls.append(a[0].shape[0]) or real(*a, **k))

    def run(least):
        monkeypatch.setattr(part, "EXPAND_MIN_NEW", least)
        eng = random_engine(small_netanex(window), seed=3, max_tokens=8192, max_seqs=8, max_context=1024)
        g = torch.Generator().manual_seed(1)
        toks = lambda n: torch.randint(0, 97, (n,), generator=g).tolist()
        logits = []
        for _ in range(4):       # the shapes are recorded at their second sight
            slots = [eng.open() for _ in range(3)]
            for lengths in ((200, 40, 333), (64, 129, 1), (1, 1, 1), (70, 33, 40), (1, 1, 1)):
                logits.append(eng.step([(s, toks(n), [n - 1]) for s, n in zip(slots, lengths)]).double().cpu())
            for s in slots:
                eng.close(s)
        assert eng.graphs.replays > 0
        return logits

    absorbed, none = run(1 << 30), len(calls)
    expanded = run(32)
    assert none == 0 and len(calls) > 0 and 1 not in calls
    for a, b in zip(absorbed, expanded):
        assert float((a - b).abs().max() / a.abs().max()) < 2e-2


@pytest.mark.parametrize("past,new,experts", [((2100,) * 5, (40,) * 5, 4), ((60,) * 9, (33, 32, 32, 32, 32, 32, 32, 32, 33), 4),
                                              ((0,), (450,), 16), ((0, 0), (20, 21), 4)])
def test_first_run_and_recording_take_the_same_form(past, new, experts, monkeypatch):
    """A shape runs eagerly at its own size until it is recorded at its bucket's: more sequences, tokens and pages.  Whether keys
    and values are expanded, and whether tokens run through their own experts only, does not change with that."""
    from burn_lm_amd.csrc import ops
    from burn_lm_amd.engine.loading import random_engine
    calls = []
    for name in ("latent_prompt", "moe_grouped"):
        monkeypatch.setattr(ops, name, lambda *a, real=getattr(ops, name), name=name, **k: calls.append(name) or real(*a, **k))
    config = small_netanex(0)
    for layer in config["layers"]:
        layer["mlp"] = dict(kind="moe", expert=dict(ff=64), router=dict(experts=experts, top=2))
    eng = random_engine(config, seed=3, max_tokens=16 * 4096, max_seqs=16, max_context=4096)
    g = torch.Generator().manual_seed(1)
    toks = lambda n: torch.randint(0, 97, (n,), generator=g).tolist()
    texts = [(toks(p), toks(n)) for p, n in zip(past, new)]
    runs, logits = [], []
    for _ in range(3):           # eagerly; eagerly, and at the bucket's size before and in the recording; replayed
        slots = [eng.open() for _ in texts]
        for s, (held, _) in zip(slots, texts):
            if held:
                eng.step([(s, held, list(range(len(held))))])        # (all rows wanted: never recorded)
        calls.clear()
        logits.append(eng.step([(s, t, [len(t) - 1]) for s, (_, t) in zip(slots, texts)]).double())
        runs.append({name: calls.count(name) for name in ("latent_prompt", "moe_grouped")})
        for s in slots:
            eng.close(s)
    assert eng.graphs.replays == 1 and sum(runs[2].values()) == 0
    assert runs[1] == {name: 3 * n for name, n in runs[0].items()}, runs
    assert float((logits[2] - logits[0]).abs().max() / logits[0].abs().max()) < 2e-2


def test_rule():
    """Few new tokens, and page tables that could name far more rows than the step has tokens, stay with the absorbed form."""
    from types import SimpleNamespace as NS

    from burn_lm_amd.parts.latent_attention import LatentAttention
    m = LatentAttention.__new__(LatentAttention)
    m.can_expand = True
    view = NS(v=torch.empty(1), page_size=64)
    q = torch.empty(64, 64, dtype=torch.bfloat16)
    rule = lambda n, B, new, after: m.expands(NS(n_seqs=B, max_len_after=after, max_new=new, n_tokens=n), q, view)
    assert rule(2048, 1, 2048, 2048) and rule(32, 1, 32, 1000) and rule(64, 2, 63, 100)
    assert not rule(1, 1, 1, 1000) and not rule(31, 1, 31, 31) and not rule(63, 2, 40, 100)
    assert rule(4096, 1, 4096, 16384) and not rule(64, 1, 64, 32768) and rule(16384, 1, 16384, 65536) and not rule(8, 8, 1, 64)
    assert not m.expands(NS(n_seqs=1, max_len_after=64, max_new=64, n_tokens=64), q[:, 1:], view)


@pytest.mark.parametrize("dtype,dim,kept", [("bfloat16", 64, True), ("float32", 64, False), ("bfloat16", 48, False)])
def test_second_layout_of_the_key_weights(dtype, dim, kept):
    """Only a part that can expand its latents keeps W_uk in both layouts."""
    from burn_lm_amd.engine.loading import random_engine
    config = small_netanex(0)
    for layer in config["layers"]:
        layer["mixer"].update(dim=dim, scale=(dim + 32) ** -0.5)
    eng = random_engine(config, seed=3, dtype=dtype, max_tokens=256, max_seqs=1, max_context=256)
    parts = [b.mixer for b in eng.model.blocks]
    assert all(m.can_expand == kept and (m.w_uk is not None) == kept for m in parts)
    slot = eng.open()
    assert bool(eng.step([(slot, list(range(90)), [89])]).isfinite().all())


def test_weights_at_any_address():
    """Weights per head that are views into larger tensors, at addresses that are no multiples of 16 bytes, give the same result."""
    from burn_lm_amd.engine.loading import random_engine
    eng = random_engine(small_netanex(0), seed=3, max_tokens=256, max_seqs=1, max_context=256)
    m, g = eng.model.blocks[0].mixer, torch.Generator().manual_seed(5)
    tensors = {name: (torch.randn(*spec.shape, generator=g) * 0.1).bfloat16().cuda() for name, spec in m.tensor_specs().items()}
    odd = lambda t: torch.cat((t.new_zeros(1), t.reshape(-1)))[1:].view(t.shape)
    slot = eng.open()
    eng.cache.reserve([(slot, 90)])
    step = eng.build_step([(slot, list(range(90)), [89])])
    x = torch.randn(90, 128, generator=g).bfloat16().cuda()
    results = []
    for form in (lambda t: t, odd):
        part = type(m)(m.params, m.names)
        part.bind({name: form(t) if name in (m.names["uk"], m.names["uv"]) else t for name, t in tensors.items()}, eng.rt)
        assert part.can_expand
        results.append(part.forward(x, step, eng.cache.views[0]).float())
    assert torch.equal(*results)


@pytest.mark.parametrize("window", [0, 100])
def test_operations_of_a_prompt(window):
    """What a step costs at the least counts the form that it runs in: written out pair by pair for a long prompt, a portion behind
    others and a single token."""
    from burn_lm_amd.parts.latent_attention import LatentAttention
    m = LatentAttention.__new__(LatentAttention)
    m.H, m.R, m.dn, m.dr, m.dv, m.window, m.can_expand = 16, 512, 128, 64, 128, window, True
    for past, new in ((0, 2048), (300, 700), (2000, 1), (0, 1)):
        see = [range(max(0, t - window + 1) if window else 0, t + 1) for t in range(past, past + new)]
        pairs, rows = sum(map(len, see)), past + new - see[0][0]
        absorbed, own = 2 * 16 * (512 + 64 + 512) * pairs, 2 * 16 * (128 + 64 + 128) * pairs
        expansion = 2 * 512 * 16 * (128 + 128)
        assert m.expanded_flops(past, new) == own + expansion * rows
        assert m.mixing_flops(past, new) == (absorbed if new == 1 and past else min(absorbed, own + expansion * (rows - new)))
        assert (m.mixing_flops(past, new) < absorbed) == (new > 1 or past == 0)
    m.can_expand = False
    assert m.mixing_flops(0, 2048) == 2 * 16 * 1088 * sum(min(t + 1, window or 2048) for t in range(2048))


def test_rule_stays_within_the_launch():
    """A sequence of more pages than a launch has rows of blocks stays with the absorbed form, however many tokens it brings."""
    from types import SimpleNamespace as NS

    from burn_lm_amd.parts.latent_attention import LatentAttention
    m = LatentAttention.__new__(LatentAttention)
    m.can_expand = True
    view, q = NS(v=torch.empty(1), page_size=64), torch.empty(64, 64, dtype=torch.bfloat16)
    rule = lambda n, after: m.expands(NS(n_seqs=1, max_len_after=after, max_new=n, n_tokens=n), q, view)
    assert rule(1 << 21, 65535 * 64) and not rule(1 << 21, 65535 * 64 + 1)
