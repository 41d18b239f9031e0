"""The narrow-row kernel's variants for any m and k (csrc/gemm_narrow_any.hip) against the oracle."""
import pytest

from test_wide_tile import _check, _inputs, _out

pytestmark = pytest.mark.gpu


def _cfg(rows, wk, u, tt):
    from tuna_amd.ops import GemmConfig

    return GemmConfig.from_dict(dict(rows_per_wave=rows, waves_m=0 if rows == 64 else 1, waves_k=wk, split_k=1, prefetch=u,
                                     x_chunk=32 * wk * u, token_tiles=tt, xcd_swizzle=0, lds_tile_rows=-5))


# the smallest operands, k below one step, one group beyond a step and before a turn's end, whole turns; a ragged last
# row tile; 1 .. 4 token tiles, several passes
@pytest.mark.parametrize("m,n,k,rows,wk,u,tt", [(8, 1, 8, 16, 16, 4, 1), (24, 4, 40, 16, 16, 2, 1), (1000, 5, 1032, 32, 8, 4, 1),
                                                (520, 16, 1016, 64, 4, 4, 1), (1192, 2, 2000, 32, 8, 8, 1), (264, 17, 4104, 32, 8, 4, 2),
                                                (72, 33, 264, 64, 4, 2, 4), (2048, 16, 4096, 64, 8, 4, 1), (1496, 64, 1096, 32, 8, 2, 2),
                                                (40, 100, 3016, 32, 8, 2, 4), (136, 30, 520, 64, 8, 2, 2)])
@pytest.mark.parametrize("epilogue", [0, 1, 2])
def test_any_shape(m, n, k, rows, wk, u, tt, epilogue):
    import torch

    from tuna_amd import _lib, ops

    cfg = _cfg(rows, wk, u, tt)
    assert "any k" in ops.describe_launch(m, n, k, cfg)
    q, s, x, code = _inputs(m, n, k, seed=m + n)
    # what lies behind x, q and the scales must not enter a sum
    x = torch.cat([x.flatten(), torch.full((4096,), float("nan"), dtype=x.dtype, device="cuda")])[:n * k].view(n, k)
    s = torch.cat([s, torch.full((64,), float("nan"), device="cuda")])[:m]
    plain = _out(n, m)
    ops.matmul(x, q, s, code, plain, m, n, k, config=cfg)
    torch.cuda.synchronize()
    _check(plain, q, s, x, code, k)
    if epilogue:
        res = torch.randn(n, m, device="cuda").half()
        fused = _out(n, m // epilogue)
        ops.matmul_fused(x, q, s, code, fused, m, n, k, epilogue, res if epilogue == _lib.EPILOGUE_RESIDUAL else None, config=cfg)
        torch.cuda.synchronize()
        p = plain.float()
        want = p + res.float() if epilogue == _lib.EPILOGUE_RESIDUAL else torch.nn.functional.silu(p[:, 0::2]) * p[:, 1::2]
        assert (fused.float() - want).abs().max() <= 4e-3 * want.abs().max() + 6e-8


# a scale per block: in LDS and too many for it, double steps beyond the last block, one and two blocks a turn, ragged rows
@pytest.mark.parametrize("m,n,k,block,rows,wk,u,tt", [(16, 1, 256, 64, 16, 16, 4, 1), (1008, 5, 1280, 64, 32, 8, 4, 1), (64, 16, 14592, 64, 64, 8, 4, 1),
                                                      (1200, 2, 2304, 128, 64, 4, 4, 1), (272, 17, 4352, 128, 32, 8, 4, 2), (144, 30, 768, 256, 64, 8, 2, 2),
                                                      (80, 64, 1536, 64, 64, 4, 2, 4), (48, 40, 22784, 64, 16, 16, 2, 1)])
def test_scale_blocks(m, n, k, block, rows, wk, u, tt):
    import torch

    from tuna_amd import ops

    q, s, x, code = _inputs(m, n, k, seed=k + n, block=block)
    out = _out(n, m)
    ops.matmul_blockwise(x, q, s, code, out, m, n, k, block, config=_cfg(rows, wk, u, tt))
    torch.cuda.synchronize()
    _check(out, q, s, x, code, k, block=block)
