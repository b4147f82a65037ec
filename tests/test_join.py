"""Products that do the work of the norm behind them: the product that joins the residual and leaves unscaled rows, the products that
read such rows, and where blocks use them.

Bounds, element by element, against 64 bits: a float sum of K products in any order is within (K + 2) u times the sum of the products'
sizes (u = 2^-24; bfloat16 operands are exact in it); rows and results stored in bfloat16 add half a place of it (2^-8)."""
import pytest
import torch

U = 2.0 ** -24
gpu = pytest.mark.gpu
SIZES = [(32, 8), (64, 64), (128, 40), (1024, 264), (2048, 512), (2048, 2048), (2560, 520), (3072, 4096), (2048, 8192), (4096, 14336), (48, 16384)]


def half_place(dtype):
    return 2.0 ** -8 if dtype == torch.bfloat16 else U


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,K", SIZES)
@pytest.mark.parametrize("M", [1, 3, 8])
def test_join(dtype, M, N, K):
    from burn_lm_amd.csrc import ops
    g = torch.Generator(device="cuda").manual_seed(M * 31 + N + K)
    columns = ops.gemv_join_columns(dtype, M, N, K)
    assert columns >= 8
    a = torch.full((M, K + 8), float("nan"), dtype=dtype, device="cuda")
    a[:, :K] = torch.randn(M, K, generator=g, device="cuda")
    a, w = a[:, :K], torch.randn(N, K, generator=g, device="cuda").to(dtype)
    h0, gamma = torch.randn(M, N, generator=g, device="cuda") * 3, torch.randn(N, generator=g, device="cuda")
    h, y = h0.clone(), torch.full((M, N), float("nan"), dtype=dtype, device="cuda")
    sums = torch.full((M, N // columns), float("nan"), device="cuda")
    ops.gemv_join(a, ops.pack_weight(w), h, gamma, y, sums, K)
    want = h0.double() + a.double() @ w.double().t()
    room = (K + 3) * U * (h0.abs().double() + a.abs().double() @ w.abs().double().t())
    assert bool(((h.double() - want).abs() <= room).all())
    scaled = want * gamma.double()
    assert bool(((y.double() - scaled).abs() <= room * gamma.abs() + half_place(dtype) * (scaled.abs() + room * gamma.abs())).all())
    squares = h.double().square().view(M, N // columns, columns).sum(-1)
    assert bool(((sums.double() - squares).abs() <= 20 * U * squares).all())


def unscaled(M, K, dtype, n, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    y, sums = torch.randn(M, K, generator=g, device="cuda").to(dtype), torch.rand(M, n, generator=g, device="cuda") * 40
    return y, sums, 1.0 / torch.sqrt(sums.double().sum(1, keepdim=True) / K + 1e-5)


def close(got, want, room, dtype):
    return bool(((got.double() - want).abs() <= room + half_place(dtype) * (want.abs() + room)).all())


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,K,n", [(16, 64, 4), (64, 128, 16), (4096, 2048, 256), (208, 2048, 252), (16384, 1024, 128), (32, 3072, 256)])
@pytest.mark.parametrize("M", [1, 3, 8])
def test_products_of_unscaled_rows(dtype, M, N, K, n):
    from burn_lm_amd.csrc import ops
    if dtype == torch.float32 and K > 2048:
        pytest.skip("the float32 kernel takes no more of K in one group")
    y, sums, inv = unscaled(M, K, dtype, n, seed=M + N)
    w = (torch.randn(N, K, device="cuda") / K ** 0.5).to(dtype)
    run = ops.gemv_mfma if dtype == torch.bfloat16 else ops.gemv_f32
    y64, w64 = y.double(), w.double()
    want, room = inv * (y64 @ w64.t()), (K + 12) * U * inv * (y64.abs() @ w64.abs().t())
    out = torch.full((M, N), float("nan"), device="cuda")
    assert close(run(y, ops.pack_weight(w), out, K, scale=(sums, 1e-5)), want, room, torch.float32)
    (g, u), (dg, du) = want.chunk(2, 1), room.chunk(2, 1)
    gated, slack = torch.nn.functional.silu(g) * u, 1.1 * dg * u.abs() + du * g.abs() + dg * du + 8 * U * (g * u).abs()
    out = torch.full((M, N // 2), float("nan"), dtype=dtype, device="cuda")
    assert close(run(y, ops.pack_weight(w, gated=True), out, K, gated=True, scale=(sums, 1e-5)), gated, slack, dtype)


@gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("K,nh,nkv,hd", [(64, 2, 1, 16), (2048, 32, 8, 64), (2048, 24, 8, 128), (3072, 24, 8, 128), (2080, 34, 4, 128),
                                         (4096, 32, 8, 128), (4096, 8, 2, 64)])
@pytest.mark.parametrize("M", [1, 8])
def test_qkv_of_unscaled_rows(dtype, M, K, nh, nkv, hd):
    """The same kernel on rows that were scaled first (and rounded once more where they are bfloat16) leaves the same queries and pages."""
    from burn_lm_amd.csrc import ops
    if dtype == torch.float32 and K > 2048:
        pytest.skip("the float32 kernel takes no more of K in one group")
    y, sums, inv = unscaled(M, K, dtype, 64, seed=K)
    y32 = (y.double() * inv).to(dtype)
    w = (torch.randn((nh + 2 * nkv) * hd, K, device="cuda") / K ** 0.5).to(dtype)
    packed, pages = ops.pack_weight(w), 2
    where = (torch.randint(0, 128, (M,), device="cuda").int(), torch.arange(M, device="cuda").int(),
             torch.arange(M * pages, device="cuda").int().view(M, pages), torch.randn(128, hd // 2, 2, device="cuda"))
    run = ops.gemv_qkv_rope if dtype == torch.bfloat16 else ops.gemv_f32_qkv_rope
    more = (0,) if dtype == torch.bfloat16 else ()
    results = []
    for x, scale in ((y, (sums, 1e-5)), (y32, None)):
        qkv = torch.zeros(M, w.shape[0], dtype=dtype, device="cuda")
        planes = torch.zeros(M * pages, nkv, 64, hd, dtype=dtype, device="cuda"), torch.zeros(M * pages, nkv, hd, 64, dtype=dtype, device="cuda")
        run(x, packed, qkv, *where, *planes, 64, nh, nkv, hd, *more, scale=scale)
        results.append([t.double() for t in (qkv, *planes)])
    # one rounding of the rows (half a place an element) and two of the results, or float sums of K products, through a turn of size |cos| + |sin|
    size = (y.double() * inv).abs() @ w.double().abs().t()
    turn = where[3].abs().sum(-1).max().item()
    room = turn * float(size.max()) * (half_place(dtype) * 2 if dtype == torch.bfloat16 else (K + 12) * 2 * U)
    for a, b in zip(*results):
        assert bool(((a - b).abs() <= room).all()) and float((a - b).norm() / b.norm()) <= (6e-3 if dtype == torch.bfloat16 else 1e-6)


@gpu
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_a_model_with_seams_and_without(dtype):
    """Prompts of a few tokens and decode steps, eager and recorded, with the norms as kernels of their own and without."""
    from burn_lm_amd.config.presets import preset
    from burn_lm_amd.engine.loading import random_engine
    config = dict(preset("llama3.2-1b"), num_hidden_layers=3)
    logits = []
    for seams in (True, False):
        engine = random_engine(config, seed=3, dtype=dtype, stored_dtype=getattr(torch, dtype), max_seqs=8, max_tokens=2048, max_context=256)
        assert engine.model.seams.count(None) == 2
        if not seams:
            engine.model.seams = [None] * len(engine.model.seams)
            for b in engine.model.blocks:
                b.inside = None
        slots = [engine.open() for _ in range(5)]
        got = [engine.step([(slots[0], [7, 8, 9], [0, 1, 2])])] + [engine.step([(s, [i + 1] * 5, [4])]) for i, s in enumerate(slots[1:])]
        for t in range(5):
            got.append(engine.step([(s, [11 * t + i], [0]) for i, s in enumerate(slots)]))
        logits.append(torch.cat(got).double())
    a, b = logits
    assert float((a - b).norm() / b.norm()) <= (1.5e-2 if dtype == "bfloat16" else 2e-6) and not torch.equal(a, b)


def test_parts_from_outside_run_as_they_are_written():
    from types import SimpleNamespace

    from burn_lm_amd.parts.attention import Attention
    from burn_lm_amd.parts.block import PreNormBlock, Seam
    from burn_lm_amd.parts.norm_rms import RMSNorm
    from burn_lm_amd.parts.swiglu import SwiGLU

    def made(cls):
        part = cls.__new__(cls)
        part.rt = SimpleNamespace(join_takes=lambda tokens, w: True)
        return part

    def sub(cls, *words):
        return type("Own" + cls.__name__, (cls,), {w: lambda self, *a, **k: None for w in words})

    def seam(front, norm, back):
        return Seam.between(made(front), made(norm), made(back))

    assert seam(Attention, RMSNorm, SwiGLU) is not None and seam(SwiGLU, RMSNorm, Attention) is not None
    assert seam(sub(Attention, "attend"), RMSNorm, sub(SwiGLU, "tensor_specs")) is not None
    for front in (sub(Attention, "forward"), sub(Attention, "output"), sub(SwiGLU, "forward"), sub(SwiGLU, "forward_after_norm")):
        assert seam(front, RMSNorm, SwiGLU) is None
    assert seam(Attention, sub(RMSNorm, "add_norm"), SwiGLU) is None
    for back in (sub(Attention, "forward"), sub(Attention, "project"), sub(SwiGLU, "forward"), sub(SwiGLU, "forward_after_norm")):
        assert seam(Attention, RMSNorm, back) is None
    patched = made(SwiGLU)
    patched.forward = lambda x, step: x
    assert Seam.between(made(Attention), made(RMSNorm), patched) is None

    def block(cls, **parts):
        b = cls(dict(dict(mixer_norm=made(RMSNorm), mixer=made(Attention), ffn_norm=made(RMSNorm), feed_forward=made(SwiGLU)), **parts))
        b.bound()
        return b

    plain, own = block(PreNormBlock), block(sub(PreNormBlock, "forward"))
    assert plain.inside is not None and plain.seam_to(plain) is not None
    assert plain.seam_to(own) is None and own.seam_to(plain) is None and plain.seam_to(object()) is None
    assert block(PreNormBlock, mixer=made(sub(Attention, "forward"))).inside is None


@gpu
@pytest.mark.parametrize("M", [2, 5, 7])
def test_rows_behind_the_last(M):
    """A tile has sixteen rows, a product of unscaled rows eight factors at most: rows behind the last, which have none, leave no trace in
    what lies behind the result, and more rows than there are factors are refused."""
    from burn_lm_amd.csrc import ops
    N, K = 96, 128
    y, sums, inv = unscaled(M, K, torch.bfloat16, 16, seed=M)
    w = torch.randn(N, K, device="cuda").bfloat16()
    for gated, columns in ((False, N), (True, N // 2)):
        packed = ops.pack_weight(w, gated=gated)
        out = torch.full((16, columns), -7.0, device="cuda")
        ops.gemv_mfma(y, packed, out[:M], K, gated=gated, scale=(sums, 1e-5))
        assert bool((out[M:] == -7.0).all()) and bool(out[:M].isfinite().all())
        more, longer, room = y.repeat(5, 1)[:9], sums.repeat(5, 1)[:9], torch.empty(9, columns, device="cuda")
        with pytest.raises(ops.KernelError):
            ops.gemv_mfma(more, packed, room, K, gated=gated, scale=(longer, 1e-5))
        with pytest.raises(ops.KernelError):
            ops.gemv_mfma(y, packed, out[:M], K, gated=gated, scale=(sums[:, :6].contiguous(), 1e-5))


@pytest.mark.parametrize("dtype,N,K,rows", [
    (torch.bfloat16, 2048, 16384, 8), (torch.bfloat16, 3072, 12288, 8), (torch.bfloat16, 4096, 14336, 8), (torch.bfloat16, 2304, 6336, 8),
    (torch.bfloat16, 2560, 10240, 8), (torch.bfloat16, 2304, 9216, 0), (torch.bfloat16, 2816, 11264, 0), (torch.bfloat16, 3584, 14336, 0),
    (torch.float32, 64, 176, 8), (torch.float32, 2048, 8192, 8), (torch.float32, 1024, 4096, 8), (torch.float32, 1152, 6336, 4),
    (torch.float32, 768, 6144, 0), (torch.float32, 1792, 14336, 4), (torch.float32, 3072, 3072, 8), (torch.float32, 3072, 8448, 0),
    (torch.float32, 2304, 12672, 0), (torch.float32, 4096, 16384, 8)])
def test_joined_where_it_is_the_shorter_way(dtype, N, K, rows):
    """The rows up to which a product is joined with the norm behind it (0: none): not where it was measured slower."""
    from burn_lm_amd.engine.runtime import Runtime
    rt = Runtime.__new__(Runtime)
    assert [rt.join_gains(dtype, M, N, K) for M in range(1, 10)] == [M <= rows for M in range(1, 10)]


class Log(list):
    def word(self, what, answer):
        return lambda *a, **k: (self.append(what), answer)[1]


def two_blocks(log):
    """Two blocks of recording parts on the CPU whose seams all hold, as a bound model has them."""
    from types import SimpleNamespace

    from burn_lm_amd.engine.model import Model
    from burn_lm_amd.parts.attention import Attention
    from burn_lm_amd.parts.base import Product
    from burn_lm_amd.parts.block import PreNormBlock
    from burn_lm_amd.parts.norm_rms import RMSNorm
    from burn_lm_amd.parts.swiglu import SwiGLU

    class Runtime:
        join_takes = lambda self, tokens, w: tokens <= 8
        join_reads = lambda self, x, w: True
        join = lambda self, *a: log.word("join", "rows")()
        linear = lambda self, *a, **k: log.word("linear", "delta")()
        gated_linear = linear

    rt = Runtime()

    def recording(cls, name, **words):
        own = dict(takes_unscaled=lambda self, tokens: True, last_weight=lambda self: None, **words)
        part = type(name, (cls,), own).__new__(type(name, (cls,), own))
        part.rt = rt
        return part

    def sublayer(cls, name):
        return recording(cls, name, forward=lambda self, *a: log.word(name + ".forward", "delta")(),
                         forward_after_norm=lambda self, *a: log.word(name + ".forward_after_norm", "delta")(),
                         forward_product=lambda self, *a: Product(log.word(name + ".forward_product", "x")(), "w"))

    def norm(name):
        return recording(RMSNorm, name, add_norm=lambda self, *a, **k: log.word(name + ".add_norm", "rows")(), joining=lambda self: ("gamma", 1e-5))

    model = Model.__new__(Model)
    model.blocks = [PreNormBlock(dict(mixer_norm=norm(f"n{i}"), mixer=sublayer(Attention, f"mixer{i}"), ffn_norm=norm(f"m{i}"),
                                      feed_forward=sublayer(SwiGLU, f"ffn{i}"))) for i in range(2)]
    for b in model.blocks:
        b.bound()
    model.seams = [None, model.blocks[0].seam_to(model.blocks[1]), None]
    model.plan = SimpleNamespace(order=[SimpleNamespace(layer=i, turn=None) for i in range(2)])
    model.entry = None
    model._embed = lambda step, copy: ("h", None)
    model.embedding = object()

    def run(tokens=3):
        del log[:]
        model.forward(SimpleNamespace(n_tokens=tokens, n_wanted=0), SimpleNamespace(views=[None, None]))
        return list(log)

    return model, rt, run


def test_parts_that_change_behind_the_binding_run_as_they_are():
    """A part, a norm, a block or a runtime that is patched or exchanged after a model was bound is called by its own words, as in steps
    of many tokens."""
    log = Log()
    joined = ["n0.add_norm", "mixer0.forward_product", "join", "ffn0.forward_product", "join", "mixer1.forward_product", "join", "ffn1.forward"]
    plain = ["n0.add_norm", "mixer0.forward", "ffn0.forward_after_norm", "n1.add_norm", "mixer1.forward", "ffn1.forward_after_norm"]
    model, rt, run = two_blocks(log)
    assert run() == joined and run(9) == plain

    model.blocks[1].mixer.forward = log.word("patched", "delta")
    assert run() == joined[:3] + ["ffn0.forward", "n1.add_norm", "patched", "ffn1.forward_after_norm"]
    model, rt, run = two_blocks(log)
    model.blocks[0].ffn_norm.add_norm = log.word("patched", "rows")
    assert run() == ["n0.add_norm", "mixer0.forward", "patched", "ffn0.forward_product"] + joined[4:]
    model, rt, run = two_blocks(log)
    model.blocks[0].feed_forward = two_blocks(log)[0].blocks[1].feed_forward
    assert run() == ["n0.add_norm", "mixer0.forward", "ffn1.forward_after_norm", "n1.add_norm"] + joined[5:]
    model, rt, run = two_blocks(log)
    model.blocks[1].forward = log.word("patched", "delta")
    assert run() == joined[:3] + ["ffn0.forward", "patched"]
    model, rt, run = two_blocks(log)
    model.blocks[0].forward = log.word("patched", "delta")
    assert run() == ["patched", "n1.add_norm"] + joined[5:]
    model, rt, run = two_blocks(log)
    model.blocks[1] = type("Own", (), dict(forward=lambda self, *a: log.word("own", "delta")()))()
    assert run() == joined[:3] + ["ffn0.forward", "own"]
    for word in ("linear", "gated_linear"):
        model, rt, run = two_blocks(log)
        setattr(rt, word, log.word("patched", "delta"))
        assert run() == plain


def test_rows_from_outside_go_through_the_plain_products():
    """Rows that a part from outside hands on in another form than the joined product reads (a stride, an address, a type) take the product
    and the norm's kernel that they took without the seam."""
    from types import SimpleNamespace

    from burn_lm_amd.engine.runtime import LinearWeight, Runtime
    rt = Runtime.__new__(Runtime)
    w = LinearWeight(torch.zeros(32, 16, dtype=torch.bfloat16))
    x = torch.zeros(4, 40, dtype=torch.bfloat16)
    assert rt.join_reads(x[:, :16], w) and rt.join_reads(x[1:, 8:24], w)
    for rows in (x[:, 1:17], x[:, ::2][:, :16], x[:, :16].float(), x.view(-1)[:144].view(4, 36)[:, :16], x[:, :16].t().contiguous().t()):
        assert not rt.join_reads(rows, w)

    log = Log()
    model, rt, run = two_blocks(log)
    type(rt).join_reads = lambda self, x, w: False
    assert run() == ["n0.add_norm", "mixer0.forward_product", "linear", "m0.add_norm", "ffn0.forward_product", "linear", "n1.add_norm",
                     "mixer1.forward_product", "linear", "m1.add_norm", "ffn1.forward"]
