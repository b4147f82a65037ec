"""Products of long prompts in tiles of 160 rows (ops.gemm_duo, fives=True), and which products run as planes of parts of tiles.

Bound: float sums of K products of bfloat16 in any order, (K + 2) 2^-24 times the sum of the products' sizes, and half a place of bfloat16
(2^-8) where the result is stored in it."""
import pytest
import torch

U = 2.0 ** -24


@pytest.mark.gpu
@pytest.mark.parametrize("groups", [0, 1, 2, 4])
@pytest.mark.parametrize("M,N,K", [(1, 8, 256), (80, 264, 512), (81, 256, 1024), (160, 512, 256), (161, 248, 1152), (319, 40, 640), (640, 2056, 1024), (1441, 304, 2048)])
def test_products(M, N, K, groups):
    from burn_lm_amd.csrc import ops
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a = torch.full((M, K + 64), float("nan"), device="cuda").bfloat16()
    a[:, :K] = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    a, w = a[:, :K], torch.randn(N, K, generator=g, device="cuda").bfloat16()
    want, room = a.double() @ w.double().t(), (K + 2) * U * (a.double().abs() @ w.double().abs().t())
    if groups == 0:
        big = torch.full((M + 1, N + 8), float("nan"), device="cuda").bfloat16()
        ops.gemm_duo(a, w, big[:M, :N], fives=True)
        assert bool(((big[:M, :N].double() - want).abs() <= room + 2.0 ** -8 * (want.abs() + room)).all())
        assert bool(big[M].isnan().all()) and bool(big[:, N:].isnan().all())
        return
    out = torch.full((groups, M, N), float("nan"), device="cuda")
    if not ops.gemm_duo_takes(a, w, out):
        with pytest.raises(ops.KernelError):
            ops.gemm_duo(a, w, out, fives=True)
        return
    assert bool(((ops.gemm_duo(a, w, out, fives=True).double().sum(0) - want).abs() <= room).all())
    with pytest.raises(ops.KernelError):
        ops.gemm_duo(a, w, out, fives=True, whole=1)


@pytest.mark.gpu
def test_a_down_projection_takes_them(monkeypatch):
    from burn_lm_amd.csrc import ops
    from burn_lm_amd.engine.runtime import Runtime
    rt, calls, real = Runtime(), [], ops.gemm_duo
    monkeypatch.setattr(ops, "gemm_duo", lambda *x, **k: (calls.append(k.get("fives", False)), real(*x, **k))[1])
    w = torch.randn(2048, 8192, device="cuda").bfloat16()
    for M, fives, groups in ((700, False, 4), (1200, True, 4), (2166, True, 2)):
        x = torch.randn(M, 8192, device="cuda").bfloat16()
        y = rt.linear(x, rt.weight(w), partials=True)
        assert calls.pop() == fives and y.shape == (groups, M, 2048) and not calls
        want, room = x.double() @ w.double().t(), 8194 * U * (x.double().abs() @ w.double().abs().t())
        assert bool(((y.double().sum(0) - want).abs() <= room).all())
        plain = rt.linear(x, rt.weight(w))          # a result that may not come as planes stays one
        assert plain.shape == (M, 2048) and not calls


def test_which_products():
    from burn_lm_amd.engine.runtime import Runtime
    rt = Runtime.__new__(Runtime)
    rt.compute_units, rt.fused_gate_up_measured = 256, True
    for M, N, K, parts in ((675, 2048, 8192, (4, False)), (1024, 2048, 8192, (4, False)), (1025, 2048, 8192, (4, True)), (1280, 2048, 8192, (4, True)),
                           (2166, 2048, 8192, (2, True)), (2560, 2048, 8192, (2, True)), (524, 4096, 14336, (4, True)), (1268, 4096, 14336, (2, True)),
                           (1281, 2048, 8192, None), (2561, 2048, 8192, None), (2048, 2048, 8192, None), (1861, 2048, 8192, None),     # halves over two groups
                           (512, 2048, 8192, None), (600, 2048, 8192, None), (2166, 2048, 4096, None), (1749, 1536, 6144, None), (9681, 3072, 8192, None)):
        assert rt.duo_part_planes(M, N, K) == parts, (M, N, K)
    rt.fused_gate_up_measured = False
    assert rt.duo_part_planes(2166, 2048, 8192) is None
