"""Fused epilogues of a launch with a balanced split: the batched persistent kernel with a batch of one, against the oracle."""
import pytest

from test_wide_tile import _check, _inputs, _out

pytestmark = pytest.mark.gpu


# whole tiles, tiles of two and of many contributors; 1, an odd number and 16 tokens; both rings
@pytest.mark.parametrize("m,n,k,waves_m,prefetch", [(256, 16, 1024, 4, 2), (1024, 1, 4096, 2, 2), (512, 7, 8192, 4, 4), (2048, 16, 14336, 1, 2),
                                                    (4096, 16, 2048, 4, 2)])
@pytest.mark.parametrize("epilogue", [1, 2])
def test_balanced_split(m, n, k, waves_m, prefetch, epilogue):
    import torch

    from tuna_amd import ops
    from tuna_amd.ops import GemmConfig

    cfg = GemmConfig.from_dict(dict(rows_per_wave=64, waves_m=waves_m, waves_k=16 // waves_m, split_k=0, prefetch=prefetch, x_chunk=1024,
                                    token_tiles=1, xcd_swizzle=1, lds_tile_rows=0))
    assert "gemm_multi_kernel" in ops.describe_launch(m, n, k, cfg)
    q, s, x, code = _inputs(m, n, k, seed=m + n)
    plain = _out(n, m)
    ops.matmul(x, q, s, code, plain, m, n, k, config=cfg)
    _check(plain, q, s, x, code, k)
    if epilogue == 1:
        res = torch.randn((n, m), dtype=torch.float16, device="cuda")
        want, out = plain.float() + res.float(), res.clone()
        ops.matmul_fused(x, q, s, code, out, m, n, k, 1, out, config=cfg)  # (in place)
    else:
        g, u = plain.float()[:, 0::2], plain.float()[:, 1::2]
        want, out = torch.nn.functional.silu(g) * u, _out(n, m // 2)
        ops.matmul_fused(x, q, s, code, out, m, n, k, 2, config=cfg)
    torch.cuda.synchronize()
    err = (out.float() - want).abs().max() / want.abs().max()
    assert err <= 4e-3, float(err)
