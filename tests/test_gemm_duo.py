"""The 256x256 product of long prompts (ops.gemm_duo): whole tiles and halves, edges in rows and columns, groups of K, gating; and the
plan that chooses between whole tiles and halves."""
import pytest
import torch


def test_plan_covers_every_tile():
    """Whole tiles and halves together are all tiles: the whole ones are all of them or full rounds; a plan is never longer than whole
    tiles alone; its fill is a share of what its rounds can hold (two halves take 1.14 of a whole tile's time)."""
    from burn_lm_amd.csrc import ops
    from burn_lm_amd.engine.runtime import DUO_HALF, duo_plan
    mixed = 0
    for gated in (False, True):
        for M in (1, 128, 129, 256, 257, 511, 512, 1000, 2048, 2166, 4097, 9681):
            for N in (8, 256, 264, 2048, 3072, 8192, 14336):
                tiles, tail = ops.gemm_duo_tiles(M, N, gated)
                columns = -(-N // (128 if gated else 256))
                assert tiles * 2 + tail >= -(-M // 128) * columns and tail in (0, columns)
                whole, rounds, fill = duo_plan(M, N, 256, gated)
                assert whole in (tiles, tiles - tiles % 256)
                mixed += 0 < whole < tiles
                if rounds <= DUO_HALF:
                    assert whole == 0 and 0 < fill <= 1 / (2 * DUO_HALF) + 1e-9
                else:
                    assert 0 < fill <= 1 + 1e-9
                assert rounds <= -(-(tiles + tail) // 256) + 1e-9
    assert mixed >= 5


def runtime():
    """A runtime's rules, for 256 units, on the CPU."""
    from burn_lm_amd.engine.runtime import Runtime
    rt = Runtime.__new__(Runtime)
    rt.compute_units, rt.fused_gate_up_measured = 256, True
    return rt


def test_plain_products_that_the_library_is_faster_with_stay_there():
    rt = runtime()
    for M, N, K, ours in ((2048, 2048, 2048, False), (3589, 2048, 2048, True), (1482, 5120, 2048, True), (2387, 3072, 3072, True), (4049, 2048, 8192, True),
                          (1856, 4096, 14336, False), (9510, 2048, 2048, True), (2735, 6144, 4096, True), (7919, 3072, 8192, True),      # one round of halves; mixed
                          (7632, 2048, 2048, False), (8183, 2048, 2048, False), (5217, 3072, 2048, False), (7999, 6144, 2048, False),    # whole rounds
                          (5326, 3072, 3072, False), (5135, 3072, 3072, False), (60, 65536, 2048, False)):
        assert rt.duo_product(M, N, K) == ours, (M, N, K)


def test_planes_that_the_library_is_faster_without():
    rt = runtime()
    for M, N, K, ours in ((2048, 2048, 8192, True), (1639, 2048, 8192, True), (1045, 3072, 8192, True), (1024, 4096, 14336, True), (1638, 2048, 6144, True),
                          (1532, 2048, 8192, False), (768, 4096, 14336, False), (2166, 2048, 8192, False), (2048, 2048, 4096, False), (2048, 2048, 2048, False),
                          (512, 8192, 8192, False)):
        assert rt.duo_planes(M, N, K) == ours, (M, N, K)


def test_projections_of_less_full_rounds_keep_their_product_and_pass():
    rt = runtime()
    for M, N, K, ours in ((2048, 3072, 2048, True), (4000, 3072, 2048, True), (2048, 5120, 3072, True), (1036, 6144, 4096, True), (9681, 5120, 3072, True),
                          (3300, 3072, 2048, False), (3356, 3072, 2048, False), (1150, 5120, 3072, False), (600, 5120, 3072, False), (256, 65536, 2048, False),
                          (2048, 10240, 8192, False)):
        assert rt.duo_qkv(M, N, K) == ours, (M, N, K)


def operands(M, N, K, gated, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(M, K + 16, generator=g).bfloat16().cuda()[:, 8:K + 8]          # rows of a wider buffer
    w = (torch.randn(N * (2 if gated else 1), K, generator=g) * K ** -0.5).bfloat16()
    w[N // 2, K - 8:] = 3.0                                                        # a wrong order of operands cannot hide
    return a, w.cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 8, 256), (128, 256, 256), (129, 264, 384), (256, 512, 256), (300, 248, 1152), (513, 1000, 384), (2100, 520, 512)])
@pytest.mark.parametrize("activation", [None, "silu", "gelu_tanh"])
def test_whole_tiles_and_halves(M, N, K, activation):
    """Every mix of whole tiles and halves gives the float64 product rounded to bfloat16 (half a step of 2^-8 of the value, and
    float32 sums: 1e-5), and the same bits."""
    from burn_lm_amd.csrc import ops
    gated = activation is not None
    a, w = operands(M, N, K, gated, M + N)
    want = a.double() @ w.double().T
    if gated:
        gate, up = want.chunk(2, 1)
        want = (torch.nn.functional.silu(gate) if activation == "silu" else torch.nn.functional.gelu(gate, approximate="tanh")) * up
    tiles, _ = ops.gemm_duo_tiles(M, N, gated)
    first = None
    for whole in sorted({0, tiles // 2, tiles}):
        big = torch.full((M, N + 8), 7.0, dtype=torch.bfloat16, device="cuda")
        ops.gemm_duo(a, w, big[:, :N], gated=gated, activation=activation or "silu", whole=whole)
        assert bool((big[:, N:] == 7.0).all())
        got = big[:, :N]
        # the gating's own float32 functions are within 2^-21 of a value of a few units
        assert float(((got.double() - want).abs() / (want.abs() + want.abs().mean())).max()) <= 2.0 ** -8
        first = got if first is None else first
        assert torch.equal(got, first)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,groups", [(300, 264, 256, 1), (257, 136, 1152, 2), (640, 256, 2048, 4)])
def test_partial_planes(M, N, K, groups):
    """Float32 planes over groups of K, the last one shorter, as whole tiles and as halves: their sum is the product to float32's sums."""
    from burn_lm_amd.csrc import ops
    a, w = operands(M, N, K, False, K)
    want = a.double() @ w.double().T
    for whole in (0, None):
        out = torch.full((groups, M, N), 7.0, device="cuda")
        ops.gemm_duo(a, w, out, whole=whole)
        assert float((out.double().sum(0) - want).abs().max() / want.abs().max()) <= 2e-6


@pytest.mark.gpu
def test_refuses_what_it_cannot_do():
    from burn_lm_amd.csrc import ops
    from burn_lm_amd.csrc.ops import KernelError
    a, w, out = (torch.zeros(n, k, dtype=torch.bfloat16, device="cuda") for n, k in ((300, 256), (264, 256), (300, 264)))
    assert ops.gemm_duo_takes(a, w, out) and not ops.gemm_duo_takes(a[:, :192], w[:, :192], out)
    assert not ops.gemm_duo_takes(a.flatten()[4:-252].view(-1, 256), w, out[:299])                  # off a multiple of 16 bytes
    assert not ops.gemm_duo_takes(a, w, torch.zeros(2, 300, 264, device="cuda"))                     # a group needs 256 of K
    for bad in (dict(whole=99), dict(whole=-1)):
        with pytest.raises(KernelError, match="whole tiles"):
            ops.gemm_duo(a, w, out, **bad)
    with pytest.raises(KernelError, match="256x256"):
        ops.gemm_mfma(a, w, out, tile=(256, 128), whole=0)
    with pytest.raises(KernelError, match="not supported"):
        ops.gemm_duo(a[:, :192], w[:, :192], out)
    with pytest.raises(KernelError, match="do not fit"):
        ops.gemm_duo(a, w[:256], out)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,plain,planes,gated", [(3600, 2048, 512, 0, None, 0), (3300, 2048, 512, None, None, 0), (2048, 2048, 6144, None, 0, None),
                                                      (1000, 8192, 256, 0, None, 0), (4300, 4096, 256, 256, None, 256)])
def test_products_of_long_prompts_take_it(monkeypatch, M, N, K, plain, planes, gated):
    """Each of the runtime's products reaches it where its plan says so, with as many whole tiles, and where not gives the same; all are
    what the plain product is."""
    from burn_lm_amd.csrc import ops
    from burn_lm_amd.engine.runtime import Runtime
    rt = Runtime(torch.bfloat16, "cuda:0")
    a, w = operands(M, N, K, False, 5)
    calls, real = [], ops.gemm_duo
    monkeypatch.setattr(ops, "gemm_duo", lambda *x, **k: (calls.append(k["whole"]), real(*x, **k))[1])
    want = a.double() @ w.double().T
    for partials, whole in ((False, plain), (True, planes if planes is not None else plain)):
        del calls[:]
        got = rt.linear(a, rt.weight(w), partials=partials)
        assert calls == ([] if whole is None else [whole]) and (got.dim() == 3) == (partials and planes is not None)
        got = got.double().sum(0) if got.dim() == 3 else got.double()
        assert float(((got - want).abs() / (want.abs() + want.abs().mean())).max()) <= 2.0 ** -8
    inner = N // 2
    gate, up = want.chunk(2, 1)
    want = torch.nn.functional.silu(gate) * up
    del calls[:]
    got = rt.gated_linear(a, rt.weight(w, gated=True))
    assert calls == ([] if gated is None else [gated])
    assert float(((got.double() - want).abs() / (want.abs() + want.abs().mean())).max()) <= 2.0 ** -7 and got.shape == (M, inner)


@pytest.mark.gpu
def test_tiles_of_256_without_halves_are_the_other_kernels(monkeypatch):
    """gemm_mfma runs its own tiles of 256x256 unless it is told how many of them are whole."""
    from burn_lm_amd.csrc import ops
    a, w = operands(300, 264, 256, False, 1)
    want, calls, real = a.double() @ w.double().T, [], ops.gemm_duo
    monkeypatch.setattr(ops, "gemm_duo", lambda *x, **k: (calls.append(k["whole"]), real(*x, **k))[1])
    for whole in (None, 0):
        got = ops.gemm_mfma(a, w, torch.empty(300, 264, dtype=torch.bfloat16, device="cuda"), tile=(256, 256), whole=whole)
        assert calls == ([] if whole is None else [0])
        assert float(((got.double() - want).abs() / (want.abs() + want.abs().mean())).max()) <= 2.0 ** -8


@pytest.mark.gpu
@pytest.mark.parametrize("whole", [0, None])
@pytest.mark.parametrize("M,K,nh,nkv,hd", [(1, 256, 2, 1, 64), (129, 384, 3, 1, 48), (257, 256, 5, 2, 128), (300, 512, 32, 8, 64), (520, 256, 1, 1, 16)])
def test_projection_with_rotation_and_pages(M, K, nh, nkv, hd, whole):
    """Heads across and inside tiles and wavefronts, a padding row, rows of many sequences at unlike places of their pages; with and
    without pages to write: as the projections of fewer rows are checked."""
    from test_kernels import _check_qkv_rope
    from burn_lm_amd.csrc import ops

    def run(x, W, out, positions, token_seq, perm, cs, kd, vd, page, write_kv):
        ops.gemm_duo_qkv_rope(x, W, out, positions, token_seq, perm, cs, kd, vd, page, nh, nkv, hd, write_kv=write_kv, whole=whole)

    _check_qkv_rope(run, "interleaved", M, K, nh, nkv, hd)


@pytest.mark.gpu
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("M,N,N2,K", [(129, 136, 8, 256), (300, 256, 264, 384), (520, 264, 512, 256)])
def test_plain_columns_beside_gated_ones(M, N, N2, K, activation):
    """A gated product with a plain one of the same rows in its launch gives the bits of the two apart, whole tiles or halves."""
    from burn_lm_amd.csrc import ops
    a, w = operands(M, 2 * N + N2, K, False, M)
    new = lambda n: torch.full((M, n), 7.0, dtype=torch.bfloat16, device="cuda")
    gated, plain = ops.gemm_duo(a, w[:2 * N], new(N), gated=True, activation=activation), ops.gemm_duo(a, w[2 * N:], new(N2))
    tiles, _ = ops.gemm_duo_tiles(M, N, True, N2)
    for whole in sorted({0, tiles // 2, tiles}):
        out, z = ops.gemm_duo_beside(a, w, new(N), new(N2), activation=activation, whole=whole)
        assert torch.equal(out, gated) and torch.equal(z, plain)
