"""Products of 17 to 64 rows whose weights are loaded past the caches: the same bits, and only for models whose weights do not stay there."""
import pytest
import torch

from burn_lm_amd.engine.runtime import LAST_LEVEL_BYTES, Runtime


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,gated,columns,groups", [(17, 8192, 2048, False, 32, 1), (64, 2056, 8200, False, 64, 4), (40, 4100, 2048, True, 64, 1), (64, 8192, 2048, False, 32, 2)])
def test_same_bits(M, N, K, gated, columns, groups):
    """Wide matrices (32 MB and more, which is where the loads differ), with columns and widths that end inside a tile."""
    from burn_lm_amd.csrc import ops
    x, w = torch.randn(M, K, device="cuda").bfloat16(), torch.randn(N * (2 if gated else 1), K, device="cuda").bfloat16()
    assert w.numel() * 2 >= 32 << 20
    shape, dtype = ((groups, M, N), torch.float32) if groups > 1 else ((M, N), torch.bfloat16)
    got = [ops.gemm_rows(x, w, torch.full(shape, 7.0, dtype=dtype, device="cuda"), gated=gated, columns=columns, once=once) for once in (False, True)]
    assert torch.equal(*got)


@pytest.mark.parametrize("layers,streams", [(1, False), (2, False), (3, True), (16, True)])
def test_models_that_stay_in_the_cache(layers, streams):
    """Layers of 122 MB: two stay from step to step, three do not; a head that is larger than the cache by itself never stays and counts for nothing."""
    rt = Runtime.__new__(Runtime)
    rt.dtype = torch.bfloat16
    rt.weight(torch.empty(128256, 2048, dtype=torch.bfloat16, device="meta"))
    for _ in range(layers):
        for n, k in ((3072, 2048), (2048, 2048), (16384, 2048), (2048, 8192)):
            rt.weight(torch.empty(n, k, dtype=torch.bfloat16, device="meta"))
    assert rt.bound_bytes == layers * 60817408 * 2 and rt.streams_weights == streams == (layers * 121634816 > LAST_LEVEL_BYTES)
