"""The tall-tile decode kernel (csrc/gemm_tall.hip): 16 RT rows x 16 NT tokens, eight waves along k, parts of k handed over
through the workspace; against the oracle."""
import pytest

from test_wide_tile import _check, _inputs, _out


def _cfg(rows, n, split):
    from tuna_amd.ops import GemmConfig

    return GemmConfig.from_dict(dict(rows_per_wave=rows, waves_m=1, waves_k=8, split_k=split, prefetch=2, x_chunk=64,
                                     token_tiles=-(-n // 16), xcd_swizzle=0, lds_tile_rows=-6))


# every tile height; one to four token tiles, the first and last count of each; fewer steps than waves (k of one step, of a
# part of one), one step more or less than a whole turn of the waves, odd and even numbers of steps per wave, k no multiple of 64
# (and no multiple of 32); parts of k with different numbers of steps; a last tile with 8, 16 and all but 8 rows missing
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,rows,split", [(32, 1, 8, 32, 1), (40, 16, 64, 32, 1), (232, 40, 1288, 32, 3), (48, 64, 512, 48, 1), (56, 33, 576, 48, 2),
                                              (1000, 17, 1096, 48, 2), (64, 49, 1024, 64, 2), (456, 32, 4160, 64, 5), (80, 5, 72, 80, 1), (792, 48, 2056, 80, 4),
                                              (96, 16, 1536, 96, 3), (680, 64, 3072, 96, 6), (112, 2, 4104, 112, 9), (1128, 61, 1984, 112, 1), (112, 30, 448, 112, 7),
                                              (128, 48, 968, 128, 2), (1160, 18, 8192, 128, 16), (264, 8, 320, 128, 1)])
@pytest.mark.parametrize("epilogue", [0, 1, 2])
def test_tiles(m, n, k, rows, split, epilogue):
    import torch

    from tuna_amd import _lib, ops

    assert f"gemm_tall_kernel<{rows} rows" in ops.describe_launch(m, n, k, _cfg(rows, n, split))
    q, s, x, code = _inputs(m, n, k, seed=m + n)
    plain, again = _out(n, m), _out(n, m)
    ops.matmul(x, q, s, code, plain, m, n, k, config=_cfg(rows, n, split))
    ops.matmul(x, q, s, code, again, m, n, k, config=_cfg(rows, n, split))
    torch.cuda.synchronize()
    assert torch.equal(plain, again)
    _check(plain, q, s, x, code, k)
    if epilogue:
        res = torch.randn(n, m, device="cuda").half()
        fused = _out(n, m // epilogue)
        ops.matmul_fused(x, q, s, code, fused, m, n, k, epilogue, res if epilogue == _lib.EPILOGUE_RESIDUAL else None, config=_cfg(rows, n, split))
        torch.cuda.synchronize()
        p = plain.float()
        want = p + res.float() if epilogue == _lib.EPILOGUE_RESIDUAL else torch.nn.functional.silu(p[:, 0::2]) * p[:, 1::2]
        # the fused output is rounded once: half of 2^-10 of it, or of fp16's step below 2^-14, which is 2^-24; the expectation
        # comes from two rounded products, 2^-11 each, the gate's through SiLU whose slope is below 1.1 (k = 8: outputs of 1e-6)
        assert (fused.float() - want).abs().max() <= 4e-3 * want.abs().max() + 2.0 ** -25


@pytest.mark.gpu
@pytest.mark.parametrize("k,rows,split", [(328, 48, 1), (1480, 112, 2), (40, 64, 1)])
def test_nothing_beyond_a_tokens_k_values_or_the_tokens_enters_a_sum(k, rows, split):
    """NaNs in front of and behind x in memory, k no multiple of 64."""
    import torch

    from tuna_amd import ops

    m, n = 224, 20
    q, s, x, code = _inputs(m, n, k, seed=3)
    big = torch.full((n * k + 16384,), float("nan"), dtype=torch.float16, device="cuda")
    big[8192:8192 + n * k] = x.reshape(-1)
    out = _out(n, m)
    ops.matmul(big[8192:8192 + n * k].view(n, k), q, s, code, out, m, n, k, config=_cfg(rows, n, split))
    torch.cuda.synchronize()
    _check(out, q, s, x, code, k)


# scales in blocks: every tile height; parts of k that start and end inside a block; a row's blocks no multiple of four; fewer
# blocks than eight waves or a wave's four; a last tile with rows missing; scales at any multiple of four bytes
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,block,rows,split", [(32, 1, 256, 64, 32, 1), (112, 20, 768, 128, 32, 2), (64, 40, 1280, 64, 48, 3), (1008, 16, 2816, 256, 48, 5),
                                                    (208, 64, 4096, 64, 64, 8), (80, 33, 1024, 64, 80, 2), (400, 9, 1792, 256, 80, 3), (592, 50, 2304, 128, 96, 7),
                                                    (112, 16, 5632, 128, 112, 1), (240, 64, 768, 64, 112, 2), (2000, 30, 4096, 64, 112, 1), (128, 48, 1536, 128, 128, 5),
                                                    (272, 3, 8192, 64, 128, 1)])
def test_scale_blocks(m, n, k, block, rows, split):
    import torch

    from tuna_amd import ops

    q, s, x, code = _inputs(m, n, k, seed=m + k, block=block)
    apart = torch.full((m * (k // block) + 8,), float("nan"), device="cuda")
    apart[1:1 + s.numel()] = s.reshape(-1)
    out, again = _out(n, m), _out(n, m)
    ops.matmul_blockwise(x, q, apart[1:1 + s.numel()].view(m, k // block), code, out, m, n, k, block, config=_cfg(rows, n, split))
    ops.matmul_blockwise(x, q, s, code, again, m, n, k, block, config=_cfg(rows, n, split))
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    _check(out, q, s, x, code, k, block=block)


@pytest.mark.parametrize("rows,n,split", [(16, 8, 1), (144, 8, 1), (40, 8, 1), (128, 64, 1), (64, 8, 0)])
def test_what_there_is_no_tile_for_is_refused(rows, n, split):
    from tuna_amd import _lib, ops

    with pytest.raises(_lib.TunaError):
        ops.validate_config(1024, n, 1024, _cfg(rows, n, split))


@pytest.mark.parametrize("k,block,split", [(256, 128, 1), (16384, 64, 1)])
def test_scale_blocks_it_has_no_room_or_loads_for_are_refused(k, block, split):
    """Two blocks a row; 256 blocks of 112 rows in LDS beside four token tiles' activations."""
    from tuna_amd import _lib, ops

    with pytest.raises(_lib.TunaError):
        ops.validate_config_blockwise(1024, 64, k, block, _cfg(112, 64, split))


def test_a_call_without_a_config_takes_it_where_it_is_predicted_to_be_faster():
    from tuna_amd import ops

    for shape in ((5120, 37, 13824), (28672, 64, 4096), (4096, 64, 14336), (8192, 24, 28672), (11008, 20, 4104)):
        assert "gemm_tall_kernel" in ops.describe_launch(*shape), shape
    for shape in ((4096, 1, 4096), (6144, 16, 4096), (4096, 64, 4096), (57344, 16, 8192), (229376, 64, 4096), (4096, 65, 14336)):
        assert "gemm_tall_kernel" not in ops.describe_launch(*shape), shape


@pytest.mark.parametrize("kind,off", [("tall", 5.1), ("tall blocks", 4.7)])
def test_the_stated_errors_are_those_of_the_kept_launches(kind, off):
    """(per cent, as stated beside tall_time in csrc/api.cpp)"""
    from test_launch_models import DATA
    from tuna_amd import launch_models as lm

    rows = [r for r in lm.read(DATA) if r["kind"] == kind]
    assert len(rows) == 440
    assert 100 * lm.errors(rows, *lm.MODELS[kind])[0] == pytest.approx(off, abs=0.06)


# (one row tile of a batched launch more than compute units; lean launches; two and three token tiles; narrow rows with two)
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,before", [(33024, 9, 1536, "weights through LDS"), (20480, 20, 8192, "weights through LDS"), (18944, 4, 3584, "gemm_lean_kernel"),
                                          (24576, 40, 3072, "weights through LDS"), (9728, 33, 3072, "gemm_lean_kernel"),
                                          (13824, 17, 5120, "gemm_narrow_kernel<LW=4")])
@pytest.mark.parametrize("epilogue", [0, 1, 2])
def test_picks_in_place_of_lean_and_batched_launches(m, n, k, before, epilogue):
    """What the library picks by itself against the general kernel: the same products, summed in another order."""
    import torch

    from tuna_amd import _lib, ops

    pick, _, instead = ops.describe_launch(m, n, k).partition(" in place of ")
    assert pick.startswith("gemm_tall_kernel") and before in instead
    general = ops.GemmConfig.from_dict(dict(rows_per_wave=64, waves_m=1, waves_k=8, split_k=1, prefetch=2, x_chunk=512, token_tiles=1,
                                            xcd_swizzle=0, lds_tile_rows=0))
    q, s, x, code = _inputs(m, n, k, seed=m + n)
    res = torch.randn(n, m, device="cuda").half()
    outs = []
    for cfg in (None, general):
        out = _out(n, m // 2 if epilogue == _lib.EPILOGUE_SILU_MUL else m)
        if epilogue:
            ops.matmul_fused(x, q, s, code, out, m, n, k, epilogue, res if epilogue == _lib.EPILOGUE_RESIDUAL else None, config=cfg)
        else:
            ops.matmul(x, q, s, code, out, m, n, k, config=cfg)
        torch.cuda.synchronize()
        outs.append(out.float())
    # (fp32 sums of the same fp16 products in another order, rounded to fp16: one unit in the last place of the largest value)
    assert (outs[0] - outs[1]).abs().max() <= 2.0 ** -10 * outs[1].abs().max()
