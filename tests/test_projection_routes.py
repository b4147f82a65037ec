"""Which products a position encoding's projection may take: the runtime's fused ones, unless the runtime brings a linear of its own."""
from types import SimpleNamespace

import pytest
import torch

from burn_lm_amd.engine.runtime import LinearWeight, Runtime
from burn_lm_amd.parts.base import Unscaled
from burn_lm_amd.parts.rope import RotaryEncoding

HEADS, KV, HD, K = 4, 2, 16, 256
FUSED = ("gemv_qkv_rope", "gemv_f32_qkv_rope", "gemm_split_qkv_rope", "gemm_rows_qkv_rope", "gemm_duo_qkv_rope")


class Recording:
    """Kernels that are asked for and not run."""

    def __init__(self, log):
        from burn_lm_amd.csrc import ops
        self.log, self.ops = log, ops

    def __getattr__(self, name):
        if name in FUSED or name == "rope_kv_write":
            return lambda *a, **k: self.log.append(name)
        return getattr(self.ops, name) if name not in ("gemm_duo_takes", "gemv_qkv_rope_supported") else lambda *a: True


def runtime(cls, log, dtype):
    rt = cls.__new__(cls)
    rt.dtype, rt.device, rt.compute_units, rt.rows_ring = dtype, torch.device("cpu"), 256, True
    rt.ops = Recording(log)
    rt.f32_qkv_packed = lambda *a: "packed"
    rt.f32_qkv_split = lambda *a: (64, 128)
    rt.duo_qkv, rt.duo_tiles = (lambda *a: True), (lambda *a: 1)
    rt.log = log
    return rt


class OwnLinear(Runtime):
    def linear(self, x, w, **k):
        self.log.append("linear")
        return torch.zeros(x.shape[0], w.w.shape[0], dtype=x.dtype)


class OwnBoth(OwnLinear):
    def qkv_plan(self, M, N, K):
        return super().qkv_plan(M, N, K)


def project(cls, M, dtype):
    log = []
    rt = runtime(cls, log, dtype)
    encoding = RotaryEncoding(dict(head_dim=HD, theta=10000.0, pairing="interleaved"), {})
    encoding.bind({}, rt)
    encoding.prepare(64, rt)
    weight = LinearWeight(torch.zeros((HEADS + 2 * KV) * HD, K, dtype=dtype), packed=torch.zeros(1))
    view = SimpleNamespace(k=torch.zeros(4, KV, 64, HD, dtype=dtype), v=torch.zeros(4, KV, HD, 64, dtype=dtype), page_size=64, store=True,
                           block_table=lambda step: torch.zeros(1, 4, dtype=torch.int32))
    step = SimpleNamespace(positions=torch.zeros(M, dtype=torch.int32), token_seq=torch.zeros(M, dtype=torch.int32), max_position=0)
    encoding.project_encode_store(torch.zeros(M, K, dtype=dtype), weight, step, view, HEADS, KV, HD)
    return log, encoding, weight


@pytest.mark.parametrize("M,dtype", [(8, torch.float32), (40, torch.float32), (500, torch.float32), (40, torch.bfloat16), (500, torch.bfloat16)])
def test_own_linear_is_called(M, dtype):
    fused = project(Runtime, M, dtype)[0]
    assert len(fused) == 1 and fused[0] in FUSED
    assert project(OwnLinear, M, dtype)[0] == ["linear", "rope_kv_write"]
    assert project(OwnBoth, M, dtype)[0] == fused


def test_own_linear_takes_no_unscaled_rows():
    for cls, takes in ((Runtime, True), (OwnLinear, False), (OwnBoth, True)):
        _, encoding, weight = project(cls, 40, torch.float32)
        encoding.rt.qkv_takes_unscaled = lambda *a: True
        assert encoding.takes_unscaled(4, weight, HEADS, KV, HD) == takes
    with pytest.raises(ValueError):
        _, encoding, weight = project(OwnLinear, 40, torch.float32)
        encoding.project_encode_store(Unscaled(torch.zeros(4, K), torch.zeros(4, 4), 1e-5), weight, None, SimpleNamespace(k=torch.zeros(1)), HEADS, KV, HD)
