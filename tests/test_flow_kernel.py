"""The decode-batch kernel (csrc/gemm_flow.hip): k-steps of all row tiles divided into shares, against the oracle."""
import pytest

from test_wide_tile import _check, _inputs, _out

pytestmark = pytest.mark.gpu


def _cfg(n, shares):
    from tuna_amd.ops import GemmConfig

    return GemmConfig.from_dict(dict(rows_per_wave=64, waves_m=4, waves_k=1, split_k=shares, prefetch=4, x_chunk=64,
                                     token_tiles=-(-n // 16), xcd_swizzle=0, lds_tile_rows=-4))


# one to four token tiles, the first and last count of each; one share, whole tiles, two and many contributors, shares that
# cross tiles; ragged last row tiles; k of one step, odd steps and units, tails that are no multiple of 64
@pytest.mark.parametrize("m,n,k,shares", [(256, 1, 64, 1), (264, 16, 256, 2), (512, 17, 1024, 2), (520, 32, 320, 1), (776, 33, 4096, 7),
                                          (1024, 48, 1288, 16), (2048, 49, 2048, 5), (1288, 64, 72, 3), (256, 64, 4104, 16),
                                          (4096, 5, 1000, 64), (640, 40, 8, 2), (8192, 16, 4096, 512)])
@pytest.mark.parametrize("epilogue", [0, 1, 2])
def test_shares(m, n, k, shares, epilogue):
    import torch

    from tuna_amd import _lib, ops

    assert "gemm_flow_kernel" in ops.describe_launch(m, n, k, _cfg(n, shares))
    q, s, x, code = _inputs(m, n, k, seed=m + n)
    plain, again = _out(n, m), _out(n, m)
    ops.matmul(x, q, s, code, plain, m, n, k, config=_cfg(n, shares))
    ops.matmul(x, q, s, code, again, m, n, k, config=_cfg(n, shares))
    torch.cuda.synchronize()
    assert torch.equal(plain, again)
    _check(plain, q, s, x, code, k)
    if epilogue:
        res = torch.randn(n, m, device="cuda").half()
        fused = _out(n, m // epilogue)
        ops.matmul_fused(x, q, s, code, fused, m, n, k, epilogue, res if epilogue == _lib.EPILOGUE_RESIDUAL else None, config=_cfg(n, shares))
        torch.cuda.synchronize()
        p = plain.float()
        want = p + res.float() if epilogue == _lib.EPILOGUE_RESIDUAL else torch.nn.functional.silu(p[:, 0::2]) * p[:, 1::2]
        assert (fused.float() - want).abs().max() <= 4e-3 * want.abs().max()


@pytest.mark.parametrize("m,n,k,block,shares", [(256, 9, 256, 64, 1), (528, 30, 1280, 64, 3), (1040, 48, 768, 128, 4), (512, 64, 4096, 64, 9),
                                                (768, 16, 1792, 256, 6)])
def test_scale_blocks(m, n, k, block, shares):
    import torch

    from tuna_amd import ops

    q, s, x, code = _inputs(m, n, k, seed=k + n, block=block)
    out = _out(n, m)
    ops.matmul_blockwise(x, q, s, code, out, m, n, k, block, config=_cfg(n, shares))
    torch.cuda.synchronize()
    _check(out, q, s, x, code, k, block=block)


def test_nothing_beyond_a_tokens_k_values_enters_a_sum():
    """NaNs behind x in memory, k no multiple of 64 and fewer steps than a unit has."""
    import torch

    from tuna_amd import ops

    m, n, k = 256, 20, 328
    q, s, x, code = _inputs(m, n, k, seed=3)
    big = torch.full((n * k + 8192,), float("nan"), dtype=torch.float16, device="cuda")
    big[:n * k] = x.reshape(-1)
    out = _out(n, m)
    ops.matmul(big[:n * k].view(n, k), q, s, code, out, m, n, k, config=_cfg(n, 2))
    torch.cuda.synchronize()
    _check(out, q, s, x, code, k)


def test_a_call_without_a_config_takes_it_where_it_is_predicted_to_be_faster():
    from tuna_amd import ops

    assert "gemm_flow_kernel" in ops.describe_launch(17920, 30, 23168)
    assert "gemm_flow_kernel" not in ops.describe_launch(6144, 16, 4096) + ops.describe_launch(57344, 16, 8192)


@pytest.mark.parametrize("m,k,counts", [(1088, 4096, (3, 0, 17, 33, 1)), (320, 1000, (64, 5, 16, 48, 20, 0, 0, 31)), (2048, 8192, (1, 16)),
                                        (512, 2048, (100, 20, 3, 70))])
def test_groups(m, k, counts):
    import numpy as np
    import torch

    from tuna_amd import ops

    offs = np.concatenate([[0], np.cumsum(counts)]).tolist()
    q, s, x, code = _inputs(m * len(counts), offs[-1], k, seed=k)
    out, again = _out(offs[-1], m), _out(offs[-1], m)
    ops.matmul_grouped(x, q, s, code, out, m, len(counts), k, offs)
    ops.matmul_grouped(x, q, s, code, again, m, len(counts), k, offs)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    for e, (lo, hi) in enumerate(zip(offs, offs[1:])):
        if hi > lo:
            _check(out[lo:hi], q, s, x[lo:hi], code, k, first_row=e * m, rows=m)
