"""Products that run beside another one of the same rows: which weights are taken, and that the results are those of the two apart."""
from types import SimpleNamespace

import pytest
import torch


def bound(part, rows, width, **fields):
    """A part with a first product of so many rows, on the CPU: what take_beside looks at."""
    from burn_lm_amd.engine.runtime import LinearWeight
    part = part.__new__(part)
    part.rt = SimpleNamespace(weight=lambda w, gated=False: LinearWeight(w, gated=gated), linear=lambda x, w: x @ w.w.T)
    for name, value in fields.items():
        setattr(part, name, value)
    part.w_in = part.w_gate_up = LinearWeight(torch.zeros(rows, width))
    return part


def test_rows_that_would_lose_their_stride_of_sixteen_bytes_stay_apart():
    from burn_lm_amd.engine.runtime import LinearWeight
    from burn_lm_amd.parts.gelu_glu import GeluGLU
    from burn_lm_amd.parts.latent_attention import LatentAttention
    from burn_lm_amd.parts.lightning import LightningAttention
    from burn_lm_amd.parts.sink_attention import SinkAttention
    for part in (GeluGLU, LatentAttention, LightningAttention, SinkAttention):
        for guest, taken in ((24, True), (20, False), (7, False)):
            p = bound(part, 64, 24, qk_norm=None)
            assert (p.take_beside(LinearWeight(torch.zeros(guest, 24))) is not None) == taken, (part, guest)
            if part is not GeluGLU:
                assert p.w_in.shape[0] == (64 + guest if taken else 64) and p.beside_at == (64 if taken else None)


def test_parts_from_outside_keep_their_own_forward():
    """Mixers and feed-forwards with a forward of their own, gates that only say gated(role, x, y), and blocks with a forward of their
    own run as they are written."""
    from burn_lm_amd.engine.runtime import LinearWeight
    from burn_lm_amd.parts.base import Gated, Part
    from burn_lm_amd.parts.gated_residual import GatedPreNormBlock, ResidualGate
    from burn_lm_amd.parts.gelu_glu import GeluGLU
    from burn_lm_amd.parts.lightning import LightningAttention

    class Mixer(LightningAttention):
        def forward(self, x, step, view):
            return 2 * x

    class FeedForward(GeluGLU):
        def forward(self, x, step):
            return 3 * x

    class Gate(Part):
        def gated(self, role, x, y):
            return Gated(y, x)

    class Block(GatedPreNormBlock):
        def forward(self, x, step, view):
            return self.gate.gated("mixer", x, self.mixer.forward(x, step, view))

    class Beside(LightningAttention):
        def forward(self, x, step, view):
            return 5 * x

        def forward_beside(self, x, step, view):
            return 5 * x, self.rt.linear(x, self.w_in)[:, self.beside_at:]

    def gate():
        g = ResidualGate.__new__(ResidualGate)
        g.weights, g.biases, g.mult, g.beside = {r: LinearWeight(torch.randn(16, 16)) for r in ("mixer", "feed_forward")}, dict(mixer=None, feed_forward=None), 1.0, set()
        g.rt = SimpleNamespace(linear=lambda x, w: x @ w.w.T)
        return g

    x = torch.randn(3, 16)
    for block in (GatedPreNormBlock, Block):
        for mixer, factor in ((Mixer, 2), (Beside, 5)):
            for g in (gate(), Gate({}, {})):
                b = block(dict(mixer_norm=None, mixer=bound(mixer, 8, 16), ffn_norm=None, feed_forward=bound(FeedForward, 32, 16), gate=g))
                want = g.weights["mixer"].w.clone() if hasattr(g, "weights") else None
                b.bound()
                if want is not None:
                    assert g.beside == ({"mixer"} if mixer is Beside else set())
                    assert g.step_flops(1) == 2 * 16 * 16 * (2 - len(g.beside))
                a = b.forward(x, None, None) if block is Block else b.run("mixer", x, None, None)
                assert torch.equal(a.y, factor * x) and torch.allclose(a.z, x if want is None else x @ want.T, atol=1e-5)
                assert torch.equal(b.run("feed_forward", x, None).y, 3 * x)


def test_columns_beside_gated_ones_fit_into_their_rounds():
    """256 units: what is left of the last round takes them, or whole tiles in place of its halves; not another round of halves."""
    from burn_lm_amd.engine.runtime import DUO_GATED_FILL, DUO_HALF, Runtime, duo_plan
    rt = Runtime.__new__(Runtime)
    rt.compute_units = 256
    for M, inner, n, taken in ((384, 8192, 2048, True), (700, 8192, 2048, True), (900, 8192, 2048, False), (1000, 8192, 2048, False), (1300, 8192, 2048, True),
                               (2048, 8192, 2048, False), (2166, 8192, 2048, True), (384, 8192, 3072, True), (1000, 8192, 512, False), (2048, 8192, 512, False),
                               (256, 65536, 2048, False)):
        assert (rt.duo_beside(M, inner, n) is not None) == taken, (M, inner, n)
    for M in range(257, 6000, 61):
        for inner, n in ((8192, 2048), (4096, 1024), (14336, 4096), (1000, 8)):
            whole = rt.duo_beside(M, inner, n)
            if whole is not None:
                alone, both = (duo_plan(M, inner, 256, True, b) for b in (0, n))
                assert whole == both[0] and alone[2] >= DUO_GATED_FILL and alone[1] <= both[1] < alone[1] + DUO_HALF


@pytest.mark.gpu
@pytest.mark.parametrize("M,together", [(384, True), (300, False), (512, False), (40, False)])
def test_feed_forward_with_its_gate_beside(monkeypatch, M, together):
    """On 8 units: gate, up and the residual's gate in one launch where the rule says so, else apart; either way the products of the
    stacked weights, rows in their order, rounded to bfloat16 (half a step of 2^-8; gate and up of the library are rounded once more in
    front of the activation, whose slope is at most 1.13)."""
    from burn_lm_amd.csrc import ops
    from burn_lm_amd.engine.runtime import Runtime
    from burn_lm_amd.parts.gelu_glu import GeluGLU
    rt = Runtime(torch.bfloat16, "cuda:0")
    rt.compute_units = 8
    K, inner, n = 256, 512, 256
    g = torch.Generator().manual_seed(M)
    matrix = lambda *shape: (torch.randn(*shape, generator=g) * shape[1] ** -0.5).bfloat16().cuda()
    x, named = torch.randn(M, K, generator=g).bfloat16().cuda(), dict(gate=matrix(inner, K), up=matrix(inner, K), down=matrix(K, inner))
    guest = matrix(n, K)
    ffn = GeluGLU(dict(width=K, inner=inner), {r: r for r in named})
    ffn.bind(named, rt)
    view = ffn.take_beside(rt.weight(guest))
    assert torch.equal(view.w, guest) and view.w.data_ptr() == ffn.stacked[2 * inner:].data_ptr()
    calls, real = [], ops.gemm_duo_beside
    monkeypatch.setattr(ops, "gemm_duo_beside", lambda *a, **k: (calls.append(k["whole"]), real(*a, **k))[1])
    gate, up = x.double() @ named["gate"].double().T, x.double() @ named["up"].double().T
    act, z = rt.gated_linear_beside(x, ffn.w_gate_up, ffn.w_beside, ffn.stacked, "gelu_tanh")
    assert calls == ([rt.duo_beside(M, inner, n)] if together else [])
    close = lambda got, want, steps: float(((got.double() - want).abs() / (want.abs() + want.abs().mean())).max()) <= steps * 2.0 ** -8
    assert close(z, x.double() @ guest.double().T, 1)
    assert close(act, torch.nn.functional.gelu(gate, approximate="tanh") * up, 1 if together else 4)
    total = lambda y: y.double().sum(0) if y.dim() == 3 else y.double()
    (y, again), plain = ffn.forward_beside(x, None), ffn.forward(x, None)
    assert torch.equal(again, z) and float((total(y) - total(plain)).norm() / total(plain).norm()) <= 2.0 ** -7


@pytest.mark.gpu
@pytest.mark.parametrize("M,together", [(512, True), (449, True), (300, False)])
@pytest.mark.parametrize("store", [True, False])
def test_projection_of_a_long_prompt_with_its_rotation(monkeypatch, M, together, store):
    """On 8 units: an encoding's projection goes through the tiles that turn and store where the rule says so; queries and pages are
    those of the product, the rotation and the write apart, which round to bfloat16 in front of the rotation as well as behind it."""
    from burn_lm_amd.csrc import ops
    from burn_lm_amd.engine.runtime import Runtime
    from burn_lm_amd.parts.base import PositionEncoding
    from burn_lm_amd.parts.rope import RotaryEncoding
    rt = Runtime(torch.bfloat16, "cuda:0")
    rt.compute_units = 8
    nh, nkv, hd, K = 6, 1, 64, 256
    g = torch.Generator().manual_seed(M)
    encoding = RotaryEncoding(dict(head_dim=hd, theta=10000.0, scaling=None, pairing="interleaved"), {})
    encoding.bind({}, rt)
    encoding.prepare(1024, rt)
    x = torch.randn(M, K, generator=g).bfloat16().cuda()
    w = rt.weight((torch.randn((nh + 2 * nkv) * hd, K, generator=g) * K ** -0.5).bfloat16().cuda())
    seq = (torch.arange(M) >= M // 3).int()                                 # two sequences, one that starts inside a page
    positions = torch.where(seq == 0, torch.arange(M) + 37, torch.arange(M) - M // 3).int().cuda()
    tables = torch.randperm(20, generator=g).int().view(2, 10).cuda()
    step = SimpleNamespace(positions=positions, token_seq=seq.cuda(), max_position=int(positions.max()), n_tokens=M, n_seqs=2)
    calls, real, out = [], ops.gemm_duo_qkv_rope, []
    monkeypatch.setattr(ops, "gemm_duo_qkv_rope", lambda *a, **k: (calls.append(k["whole"]), real(*a, **k))[1])
    for apart in (False, True):
        k, v = torch.zeros(20, nkv, 64, hd, dtype=torch.bfloat16, device="cuda"), torch.zeros(20, nkv, hd, 64, dtype=torch.bfloat16, device="cuda")
        view = SimpleNamespace(k=k, v=v, page_size=64, store=store, block_table=lambda step: tables)
        run = PositionEncoding.project_encode_store if apart else RotaryEncoding.project_encode_store
        out.append((run(encoding, x, w, step, view, nh, nkv, hd)[:, :nh * hd], k, v))
        assert calls == ([rt.duo_tiles(M, 512)] if together else [])
    # apart, a pair (u, v) is rounded in front of its rotation: 2^-8 (|u c| + |v s|), at most 2^-8 of the pair's length, which turning
    # keeps; both round their results, 2^-8 each; 2 % for the roundings' own sizes and the sums' order
    for i, (a, b) in enumerate(zip(*out)):
        a, b = a.double(), b.double()
        length = b.unflatten(-1, (-1, 2)).norm(dim=-1).repeat_interleave(2, -1) if i < 2 else 0.0
        assert bool(((a - b).abs() <= 1.02 * 2.0 ** -8 * (length + 2 * b.abs())).all())
    assert bool(out[0][1].any()) == store and bool(out[0][2].any()) == store
