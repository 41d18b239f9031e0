"""The broad-tile kernel (csrc/gemm_broad.hip): two row groups of 16 RT rows, four k groups, 64 / 80 / 96 tokens a tile, activations
through LDS without registers; against the oracle."""
import pytest

from test_wide_tile import _check, _inputs, _out


def _cfg(rows, tokens, split):
    from tuna_amd.ops import GemmConfig

    return GemmConfig.from_dict(dict(rows_per_wave=rows, waves_m=2, waves_k=4, split_k=split, prefetch=2, x_chunk=256,
                                     token_tiles=tokens // 16, xcd_swizzle=0, lds_tile_rows=-7))


# every tile height and width; one unit of four steps, two, three; fewer steps than a unit, units that k does not fill, k no
# multiple of 64; a last tile of rows with 8 and all but 8 missing; one token, a last token tile with one and all but one;
# parts of k with different numbers of units
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,rows,tokens,split", [(64, 1, 8, 64, 64, 1), (72, 65, 256, 64, 64, 1), (120, 96, 520, 64, 96, 1), (1000, 81, 1096, 64, 80, 2),
                                                     (96, 64, 768, 96, 64, 1), (184, 80, 2056, 96, 80, 3), (1048, 191, 1280, 96, 96, 4), (104, 128, 320, 96, 64, 1),
                                                     (128, 96, 1024, 128, 96, 1), (136, 97, 4104, 128, 96, 5), (1400, 160, 1984, 128, 80, 1), (248, 300, 576, 128, 64, 2),
                                                     (256, 70, 72, 128, 80, 1), (640, 66, 8192, 128, 80, 16),
                                                     (160, 96, 1544, 160, 96, 2), (312, 100, 1024, 160, 64, 3), (168, 79, 64, 160, 80, 1), (960, 85, 2048, 192, 80, 4),
                                                     (200, 64, 840, 192, 64, 1), (256, 130, 3000, 256, 64, 2), (1272, 64, 4096, 256, 64, 9), (264, 33, 520, 256, 64, 1)])
@pytest.mark.parametrize("epilogue", [0, 1, 2])
def test_tiles(m, n, k, rows, tokens, split, epilogue):
    import torch

    from tuna_amd import _lib, ops

    cfg = _cfg(rows, tokens, split)
    assert f"gemm_broad_kernel<{rows} rows x {tokens} tokens" in ops.describe_launch(m, n, k, cfg)
    q, s, x, code = _inputs(m, n, k, seed=m + n)
    plain, again = _out(n, m), _out(n, m)
    ops.matmul(x, q, s, code, plain, m, n, k, config=cfg)
    ops.matmul(x, q, s, code, again, m, n, k, config=cfg)
    torch.cuda.synchronize()
    assert torch.equal(plain, again)
    _check(plain, q, s, x, code, k)
    if epilogue:
        res = torch.randn(n, m, device="cuda").half()
        fused = _out(n, m // epilogue)
        ops.matmul_fused(x, q, s, code, fused, m, n, k, epilogue, res if epilogue == _lib.EPILOGUE_RESIDUAL else None, config=cfg)
        torch.cuda.synchronize()
        p = plain.float()
        want = p + res.float() if epilogue == _lib.EPILOGUE_RESIDUAL else torch.nn.functional.silu(p[:, 0::2]) * p[:, 1::2]
        # (one rounding of the output - 2^-11 of it, 2^-25 below fp16's normal range - and the two of the product it is made from)
        assert (fused.float() - want).abs().max() <= 4e-3 * want.abs().max() + 2.0 ** -25


@pytest.mark.gpu
@pytest.mark.parametrize("k,rows,tokens,split", [(328, 64, 64, 1), (1480, 128, 96, 2), (40, 96, 80, 1)])
def test_nothing_beyond_a_tokens_k_values_or_the_tokens_enters_a_sum(k, rows, tokens, split):
    """NaNs in front of and behind x in memory, k no multiple of 64."""
    import torch

    from tuna_amd import ops

    m, n = 224, 70
    q, s, x, code = _inputs(m, n, k, seed=3)
    big = torch.full((n * k + 16384,), float("nan"), dtype=torch.float16, device="cuda")
    big[8192:8192 + n * k] = x.reshape(-1)
    out = _out(n, m)
    ops.matmul(big[8192:8192 + n * k].view(n, k), q, s, code, out, m, n, k, config=_cfg(rows, tokens, split))
    torch.cuda.synchronize()
    _check(out, q, s, x, code, k)


# parts of k that start and end inside a block; a row's blocks no multiple of four
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,block,rows,tokens,split", [(64, 70, 256, 64, 64, 80, 1), (112, 64, 768, 128, 64, 64, 2), (208, 128, 2304, 64, 96, 64, 3),
                                                           (400, 90, 1792, 256, 96, 80, 2), (128, 65, 4096, 64, 128, 80, 2), (1008, 100, 2816, 256, 128, 64, 3), (336, 96, 1024, 128, 160, 64, 2), (176, 70, 2560, 64, 192, 80, 3),
                                                           (528, 65, 3840, 64, 256, 64, 4), (272, 90, 14336, 64, 128, 80, 1), (192, 64, 2048, 1024, 96, 64, 2),
                                                           (512, 80, 1536, 512, 192, 80, 1)])
def test_scale_blocks(m, n, k, block, rows, tokens, split):
    import torch

    from tuna_amd import ops

    q, s, x, code = _inputs(m, n, k, seed=m + k, block=block)
    apart = torch.full((m * (k // block) + 8,), float("nan"), device="cuda")
    apart[1:1 + s.numel()] = s.reshape(-1)
    out, again = _out(n, m), _out(n, m)
    ops.matmul_blockwise(x, q, apart[1:1 + s.numel()].view(m, k // block), code, out, m, n, k, block, config=_cfg(rows, tokens, split))
    ops.matmul_blockwise(x, q, s, code, again, m, n, k, block, config=_cfg(rows, tokens, split))
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    _check(out, q, s, x, code, k, block=block)


@pytest.mark.parametrize("rows,tokens,split", [(32, 64, 1), (224, 64, 1), (80, 64, 1), (192, 96, 1), (256, 80, 1), (128, 48, 1), (128, 112, 1), (64, 64, 0)])
def test_what_there_is_no_tile_for_is_refused(rows, tokens, split):
    from tuna_amd import _lib, ops

    with pytest.raises(_lib.TunaError):
        ops.validate_config(1024, 100, 1024, _cfg(rows, tokens, split))


# groups of one to several token tiles, empty ones among them, one token more or less than a tile's; rows no multiple of any
# tile's; k no multiple of a unit or of 64
@pytest.mark.gpu
@pytest.mark.parametrize("m,k,counts", [(2048, 1408, (65, 64, 96, 97, 33, 0, 80, 81, 70, 1, 128, 66, 90, 72, 0, 100)), (1088, 4096, (70, 90, 40, 88, 96, 66, 71, 80)),
                                        (4992, 1000, (64, 0, 0, 161, 5, 76, 95, 77)), (4096, 2056, (33, 48, 64, 60, 50, 41, 64, 63, 59, 37, 62, 64)),
                                        (14336, 512, (0, 66, 79, 0))])
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


def test_a_call_without_a_config_takes_it_where_it_is_predicted_to_be_faster():
    from tuna_amd import ops

    for shape in ((28672, 80, 4096), (8192, 160, 8192), (4096, 256, 14336), (5120, 96, 13824), (57344, 64, 8192)):
        assert "gemm_broad_kernel" in ops.describe_launch(*shape), shape
    for shape in ((4096, 100, 4096), (4096, 48, 14336), (28672, 513, 4096), (57344, 512, 8192), (8192, 64, 8192)):
        assert "gemm_broad_kernel" not in ops.describe_launch(*shape), shape


def test_256_x_256_tiles_stay_where_their_price_is_known_to_be_too_high():
    """Tiles of both kinds over long k, and four parts and more with scale blocks: broad tiles take 1.13 x and 1.14 x the time there."""
    from tuna_amd import ops

    for shape in ((8192, 384, 28672), (7744, 331, 24256), (16064, 264, 23704)):
        assert ops.describe_launch(*shape).startswith("gemm_wide_kernel"), shape
    for shape in ((12672, 254, 13056, 128), (15552, 229, 23040, 128), (8064, 355, 24064, 64)):
        c, _hit = ops.select_config_blockwise(*shape)
        assert (c.lds_tile_rows, c.token_tiles) == (256, 16), shape


@pytest.mark.parametrize("kind,off", [("broad", 4.9), ("broad blocks", 4.4)])
def test_the_stated_errors_are_those_of_the_kept_launches(kind, off):
    """(per cent, as stated beside broad_time in csrc/api.cpp)"""
    from test_launch_models import DATA
    from tuna_amd import launch_models as lm

    rows = [r for r in lm.read(DATA) if r["kind"] == kind]
    assert len(rows) == 440
    assert 100 * lm.errors(rows, *lm.MODELS[kind])[0] == pytest.approx(off, abs=0.06)
