"""Latent attention of decode steps cut into pieces of half pages: the four wavefronts of a block share a piece's lanes, some of which do
not go round in four, and some sizes leave a wavefront without any.

Bound, elementwise: the probabilities and the results' factors are rounded to bfloat16 (2^-9 each way of the weights, 2^-8 in all with
their sum's), on values that the largest of a column bounds; scores are float sums of R + Dr products, (R + Dr) 2^-24 of at most 40."""
import types

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("R,Dr", [(512, 64), (384, 64), (160, 32), (96, 16), (48, 16), (32, 16), (32, 8)])
@pytest.mark.parametrize("H,window", [(16, 0), (5, 0), (20, 45)])
def test_pieces(R, Dr, H, window):
    from burn_lm_amd.csrc import ops
    dev, lengths = "cuda", (1, 31, 32, 33, 130, 257)
    g = torch.Generator(device=dev).manual_seed(R + H)
    B, P = len(lengths), 5
    keys = torch.full((B * P, 1, 64, R + Dr), float("nan"), device=dev).bfloat16()
    rows = torch.randn(B, P * 64, R + Dr, generator=g, device=dev).bfloat16()
    table = torch.randperm(B * P, generator=g, device=dev).int().view(B, P)
    for b, n in enumerate(lengths):                 # places past the data hold no number
        for i in range(n):
            keys[int(table[b, i // 64]), 0, i % 64] = rows[b, i]
    values = keys[..., :R].transpose(2, 3).contiguous()
    q = torch.randn(B, H, R + Dr, generator=g, device=dev).bfloat16()
    sinks = torch.randn(H, generator=g, device=dev)
    step = types.SimpleNamespace(cu_seqlens=torch.arange(B + 1, device=dev).int(), lens_after=torch.tensor(lengths, device=dev).int(),
                                 n_seqs=B, max_new=1, n_tokens=B)
    scale = (R + Dr) ** -0.5
    for pieces in (2, 3, 9, 64):
        for s in (None, sinks):
            got = torch.empty(B, H, R, device=dev)
            ops.latent_attn_mfma(q, got, keys, values, step, table, 64, H, R, Dr, scale, pieces, window=window, sinks=s)
            for b, n in enumerate(lengths):
                k = rows[b, max(0, n - window) if window else 0: n].double()
                scores = scale * (q[b].double() @ k.T)
                if s is not None:
                    scores = torch.cat([scores, s.double()[:, None]], 1)
                want = torch.softmax(scores, 1)[:, :k.shape[0]] @ k[:, :R]
                room = 2.0 ** -8 + 2 * (R + Dr) * 2.0 ** -24 * 40
                assert float((got[b].double() - want).abs().max()) <= room * float(k[:, :R].abs().max()), (b, pieces)


def test_most_pieces():
    """Wide latents: a block for every unit, up to four pieces from a block for every fourth unit on; narrow ones: four blocks for every unit."""
    from burn_lm_amd.parts.latent_attention import most_pieces
    tiles = (1, 8, 16, 64, 90, 200, 300, 1024, 1025)
    assert [most_pieces(n, 512, 256) for n in tiles] == [64, 32, 16, 4, 4, 4, 3, 1, 0]
    assert [most_pieces(n, 192, 256) for n in tiles] == [64, 64, 64, 16, 11, 5, 3, 1, 0]
