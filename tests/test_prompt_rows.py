"""What lies between a prompt's projections and its attention, eight lanes at a time, against the same rows in calls of few, which go
element by element (the rule that chooses is told which it is, here): norms of heads and of rows, rotation in either pairing, latents, and the pages.  Sums of squares
are added in another order there, so a normed value may be rounded to the neighbouring bfloat16 (2^-8 of it); all else is the same."""
from types import SimpleNamespace

import pytest
import torch

PS = 64


@pytest.fixture(autouse=True)
def by_length(request, monkeypatch):
    """Calls of more than 60 rows take the wide kernels where they can, others never."""
    if "gpu" in request.keywords:
        from burn_lm_amd.csrc import ops
        monkeypatch.setattr(ops, "wide_rows", lambda kind, T, step: T > 60)


def test_tokens_of_many_sequences_keep_the_kernels_that_are_faster_for_them():
    """Steps of a token or a few of every sequence go token by token up to where the wide kernels were measured to be ahead; runs of
    eight and more sooner; a shape that is recorded goes by its bucket."""
    from burn_lm_amd.csrc import ops
    step = lambda seqs, bucket=None: SimpleNamespace(n_seqs=seqs, bucket=bucket)
    for kind, runs, few in (("heads", 65, 384), ("rows", 65, 128), ("turns", 65, 65), ("latents", 384, 1024)):
        assert ops.wide_rows(kind, runs, step(runs // 8)) and not ops.wide_rows(kind, runs - 1, step(1))
        for each in (1, 7):
            assert ops.wide_rows(kind, few, step(-(-few // each))) and not ops.wide_rows(kind, few - 1, step(-(-few // each)))
        assert ops.wide_rows(kind, 3, step(1, (2048, 4, 4096))) and not ops.wide_rows(kind, 4000, step(1, (64, 64, 4096)))


def steps(T, few):
    """Tokens of three sequences that start in the middle of their pages, one of them padding at its end; whole, and in pieces."""
    n = [T // 2 + 3, T // 3, 0]
    n[2] = T - sum(n)
    past = [0, 61, 130]
    seq = torch.repeat_interleave(torch.arange(3), torch.tensor(n)).int()
    pos = torch.cat([torch.arange(p, p + k) for p, k in zip(past, n)]).int()
    seq[-2:] = -1
    top = int(pos.max())
    make = lambda a, b: SimpleNamespace(n_tokens=b - a, positions=pos[a:b].contiguous().cuda(), token_seq=seq[a:b].contiguous().cuda(), max_position=top)
    pages = -(-(top + 1) // PS)
    tables = torch.randperm(3 * pages, generator=torch.Generator().manual_seed(T)).view(3, pages).int().cuda()
    return make(0, T), [(a, min(T, a + few), make(a, min(T, a + few))) for a in range(0, T, few)], tables


def close(a, b):
    assert bool(((a.float() - b.float()).abs() <= b.float().abs() * 2.0 ** -7).all())


def table_of(rot, positions):
    angle = torch.arange(positions)[:, None].double() * 50.0 ** (-2.0 * torch.arange(rot // 2).double() / rot)
    return torch.stack((angle.cos(), angle.sin()), -1).float().cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["heads", "rows", "maps"])
@pytest.mark.parametrize("T,H,G,dk,dv,bias", [(65, 4, 2, 64, 128, True), (130, 6, 2, 8, 24, False), (300, 2, 2, 512, 512, True), (97, 40, 4, 128, 64, True)])
def test_norms(mode, T, H, G, dk, dv, bias):
    from burn_lm_amd.csrc import ops
    g = torch.Generator().manual_seed(T)
    whole, parts, tables = steps(T, 60)
    Gv = G // 2 if mode == "maps" else G
    need = (H + G) * dk + Gv * dv
    rows = torch.randn(T, need + 8, generator=g).bfloat16().cuda()
    b = torch.randn(need, generator=g).cuda() if bias else None
    qw, kw = ((torch.rand(n * dk if mode == "rows" else dk, generator=g) + 0.5).cuda() if bias else None for n in (H, G))
    out = []
    for pieces in ([(0, T, whole)], parts):
        kc = torch.zeros(tables.numel(), Gv, PS, dk * (G // Gv), dtype=torch.bfloat16, device="cuda")
        vc = torch.zeros(tables.numel(), Gv, dv, PS, dtype=torch.bfloat16, device="cuda")
        x = rows.clone()
        q = torch.full((T, 2 * H * dk), 9.0, dtype=torch.bfloat16, device="cuda") if mode == "maps" else None
        for a, e, step in pieces:
            ops.qkv_norm(x[a:e], b, qw, kw, 0.1, step, tables, kc, vc, PS, H, G, dk, dv, whole_rows=mode == "rows", growth=(0.7, 20),
                         q_out=q[a:e] if q is not None else None)
        out.append((x, kc, vc, q if q is not None else x))
    close(out[0][0], out[1][0])
    close(out[0][1], out[1][1])
    close(out[0][3], out[1][3])
    assert torch.equal(out[0][2], out[1][2]) and torch.equal(out[0][0][:, H * dk:], rows[:, H * dk:])


@pytest.mark.gpu
@pytest.mark.parametrize("adjacent", [False, True])
@pytest.mark.parametrize("T,H,G,dk,dv,rot,store,same", [(65, 4, 2, 128, 64, 64, True, False), (200, 3, 1, 40, 8, 16, True, False),
                                                        (90, 2, 2, 64, 64, 64, True, True), (130, 5, 2, 24, 16, 0, True, False),
                                                        (70, 4, 2, 128, 64, 32, False, False)])
def test_rotation(adjacent, T, H, G, dk, dv, rot, store, same):
    from burn_lm_amd.csrc import ops
    g = torch.Generator().manual_seed(T)
    whole, parts, tables = steps(T, 60)
    need = H * dk + (G * (dk + (0 if same else dv)) if store else 0)
    rows = torch.randn(T, need + 16, generator=g).bfloat16().cuda()
    bias, scale = torch.randn(need, generator=g).cuda(), (torch.rand(H, generator=g) + 0.5).cuda()
    cs = table_of(rot, whole.max_position + 1) if rot else None
    out = []
    for pieces in ([(0, T, whole)], parts):
        kc = torch.zeros(tables.numel(), G, PS, dk, dtype=torch.bfloat16, device="cuda")
        vc = torch.zeros(tables.numel(), G, dv, PS, dtype=torch.bfloat16, device="cuda")
        x = rows.clone()
        for a, e, step in pieces:
            ops.qkv_prepare(x[a:e], bias, cs, rot, step, tables if store else None, kc if store else None, vc if store else None, PS, H, G, dk, dv,
                            write_kv=store, adjacent=adjacent, values_are_keys=same, q_scale=scale)
        out.append((x, kc, vc))
    close(out[0][0], out[1][0])
    close(out[0][1], out[1][1])
    assert torch.equal(out[0][2], out[1][2]) and bool(out[0][2].any()) == store


@pytest.mark.gpu
@pytest.mark.parametrize("adjacent", [False, True])
@pytest.mark.parametrize("T,H,dn,dr,R,rot,absorbed,pages,store",
                         [(65, 4, 128, 64, 512, 64, False, True, True), (130, 3, 8, 16, 40, 16, True, True, True),
                          (90, 16, 64, 32, 480, 16, True, False, True),           # no transposed pages, a quarter of the lanes a block
                          (97, 2, 16, 32, 504, 32, False, False, True),           # the same, units that end inside a wavefront
                          (70, 5, 128, 64, 504, 64, True, True, True),
                          (130, 4, 24, 64, 512, 32, False, True, False),          # another layer's rows: the queries alone
                          (70, 2, 128, 64, 960, 64, False, True, True)])          # latents beyond the wide kernel: token by token both times
def test_latents(adjacent, T, H, dn, dr, R, rot, absorbed, pages, store):
    from burn_lm_amd.csrc import ops
    g = torch.Generator().manual_seed(T)
    whole, parts, tables = steps(T, 60)
    down = torch.randn(T, R + dr + 8, generator=g).bfloat16().cuda()[:, :R + dr]
    q = torch.randn(T, H * (dn + dr), generator=g).bfloat16().cuda()
    w, cs = (torch.rand(R, generator=g) + 0.5).cuda(), table_of(rot, whole.max_position + 1)
    for dtype in (torch.bfloat16, torch.float32):
        out = []
        for pieces in ([(0, T, whole)], parts):
            kc = torch.zeros(tables.numel(), 1, PS, R + dr, dtype=torch.bfloat16, device="cuda")
            vc = torch.zeros(tables.numel(), 1, R, PS, dtype=torch.bfloat16, device="cuda")
            turned = torch.zeros(T, H, R + dr if absorbed else dr, dtype=dtype, device="cuda")
            for a, e, step in pieces:
                ops.latent_write(down[a:e] if store else None, q[a:e], w, 1e-5, cs, rot, turned[a:e], kc, step, tables, PS, H, dn, R, dr,
                                 write_kv=store, vcache=vc if pages else None, adjacent=adjacent)
            out.append((kc, vc, turned))
        for x, y in zip(*out):
            close(x, y) if dtype == torch.bfloat16 or x.dtype == torch.bfloat16 else torch.testing.assert_close(x, y, rtol=2e-6, atol=2e-6)
        assert bool(out[0][0].any()) == store and bool(out[0][1].any()) == (pages and store) and bool(out[0][2].any())
        assert torch.equal(out[0][0][..., :R].transpose(2, 3)[out[0][1] != 0], out[0][1][out[0][1] != 0])
