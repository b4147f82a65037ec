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
