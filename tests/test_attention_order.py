"""The order in which a float32 prompt's blocks start: every place of every key-value head once, and the two blocks that a compute unit works on at
once far apart in length, however many heads there are."""
import pytest

from burn_lm_amd.csrc import ops


@pytest.mark.parametrize("units", [256, 80, 1])
@pytest.mark.parametrize("nkv", [1, 2, 3, 4, 8, 12, 16, 32, 300])
@pytest.mark.parametrize("blocks", [1, 7, 64, 130, 257])
def test_every_place_once(nkv, units, blocks):
    places = [[] for _ in range(nkv)]
    for at in range(blocks * nkv):
        places[at % nkv].append(ops.attn_prefill_f32_place(at, blocks, nkv, units))
    assert all(sorted(p) == list(range(blocks)) for p in places)


@pytest.mark.parametrize("nkv", [1, 2, 4, 8, 16, 32])
def test_long_beside_short(nkv):
    """Two whole runs a head: the places of the blocks at and at + units add up to the same for every block."""
    units = 256
    blocks = 2 * units // nkv
    sums = {ops.attn_prefill_f32_place(at, blocks, nkv, units) + ops.attn_prefill_f32_place(at + units, blocks, nkv, units) for at in range(units)}
    assert sums == {blocks - 1}
