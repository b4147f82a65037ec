"""Products that run beside another one of the same rows: which weights are taken, and that the results are those of the two apart."""
from types import SimpleNamespace

import pytest
import torch


def bound(part, rows, width, **fields):
    """A part with a first product of so many rows, on the CPU: what take_beside looks at."""
    from burn_lm_amd.engine.runtime import LinearWeight
    part = part.__new__(part)
    part.rt = SimpleNamespace(weight=lambda w, gated=False: LinearWeight(w, gated=gated))
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
            assert p.take_beside(LinearWeight(torch.zeros(guest, 24))) == taken, (part, guest)
            if part is not GeluGLU:
                assert p.w_in.shape[0] == (64 + guest if taken else 64) and p.beside_at == (64 if taken else None)
