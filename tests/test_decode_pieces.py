"""Pieces of a decode attention's key range for wide heads: down to one page per wavefront while the pieces run in one round
and are no more than eight."""


def test_wide_heads():
    from burn_lm_amd.parts.attention import decode_splits
    assert [decode_splits(18, blocks, 128) for blocks in (32, 64, 80, 128, 129, 256)] == [5, 4, 3, 2, 1, 1]
    assert [decode_splits(pages, 32, 128) for pages in (16, 17, 24, 32, 48)] == [4, 5, 6, 8, 8]
    assert [decode_splits(pages, 16, 128) for pages in (32, 48, 64, 100)] == [8, 8, 8, 12]      # no more than eight by this rule
    assert [decode_splits(18, blocks, 64) for blocks in (32, 64, 80)] == [4, 2, 2]       # narrow heads as before
    for pages in (9, 17, 33, 100):
        for blocks in (4, 24, 40, 72, 200):
            n = decode_splits(pages, blocks, 128)
            assert 1 <= n <= 32 and (n == 1 or blocks * n <= 256 or n <= -(-128 // blocks)) and pages // n >= 2
