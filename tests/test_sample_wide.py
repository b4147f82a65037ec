"""Nucleus draws by blocks of 1,024 threads, which list the weights of the first level's bin, against the same row drawn alone (blocks of
256 threads, a histogram to each level): the masses are whole numbers and the kept ones are summed chunk by chunk in the same order, so
the tokens are the same."""
import pytest
import torch


def rows_of(kind, R, V, g):
    z = torch.randn(R, V, generator=g, device="cuda")
    if kind == "normal":
        return z * 1.5
    if kind == "flat":                       # all in one bin: more than a list holds
        return torch.zeros_like(z)
    if kind == "narrow":                     # lists of some rows, some slices, are full
        return z * torch.linspace(0.0, 0.4, R, device="cuda")[:, None]
    if kind == "part":                       # some of a row's slices have more in the bin than a list holds, the others an entry or none
        z = torch.where(torch.arange(V, device="cuda") < torch.arange(R, device="cuda")[:, None] * V // R, z * 0.002, z - 9.0)
        return z.roll(V // 3, 1)
    if kind == "ties":                       # few different weights
        return (z * 2.0).round()
    z[:, V // 3:] = -float("inf")            # masked: slices without any mass, one with a single token
    z[0] = -float("inf")
    z[0, V - 1] = 3.0
    return z


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["normal", "flat", "narrow", "part", "ties", "masked"])
@pytest.mark.parametrize("R,V,ld", [(16, 98304, 98304), (33, 50021, 50021), (64, 49153, 49156), (64, 128256, 128256), (100, 32000, 32000),
                                    (128, 24578, 24578)])
def test_draws_are_those_of_a_row_alone(kind, R, V, ld):
    from burn_lm_amd.csrc import ops
    g = torch.Generator(device="cuda").manual_seed(R + V)
    z = torch.full((R, ld), float("nan"), device="cuda")
    z[:, :V] = rows_of(kind, R, V, g)
    z = z[:, :V]
    for temperature, top_p in ((0.8, 0.9), (1.3, 0.05), (0.3, 0.999)):
        u = torch.rand(R, generator=g, device="cuda")
        u[0], u[1] = 0.0, 1.0 - 2.0 ** -24
        together = ops.sample(z, u, temperature, top_p)
        alone = torch.cat([ops.sample(z[i:i + 1], u[i:i + 1], temperature, top_p) for i in range(R)])
        assert torch.equal(together, alone)
        assert torch.equal(together, ops.sample(z, u, temperature, top_p))
        assert bool(z.gather(1, together.long()[:, None]).isfinite().all())
