"""256-row tiles of any width (csrc/gemm_wide.hip, csrc/gemm_wide_whole.hip): every number of token tiles, whole, split and shared; the
epilogues; scale blocks exchanged between lanes; groups of several widths in one launch; the picks and their model."""
import ctypes
import os
import re
import shutil
import subprocess

import numpy as np
import pytest

from test_wide_tile import _cfg as _cfg256
from test_wide_tile import _check, _inputs, _out


def _cfg(token_tiles, split):
    from tuna_amd.ops import GemmConfig

    return GemmConfig.from_dict(dict(rows_per_wave=64, waves_m=token_tiles, waves_k=1, split_k=split, prefetch=2, x_chunk=64, token_tiles=16,
                                     xcd_swizzle=0, lds_tile_rows=256))


# every number of token tiles, full and with a ragged last one, one to several tiles of tokens, odd and even numbers of steps, k tails, rows
# that no tile divides
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,token_tiles,split", [(256, 128, 64, 8, 1), (264, 100, 192, 8, 1), (520, 158, 128, 10, 1), (256, 315, 320, 10, 1),
                                                     (512, 177, 256, 12, 1), (264, 383, 72, 12, 1), (256, 223, 448, 14, 1), (776, 660, 200, 14, 1),
                                                     (256, 256, 128, 16, 1), (1032, 500, 1000, 16, 1), (264, 129, 8, 16, 1),
                                                     (264, 130, 192, 9, 1), (256, 288, 64, 9, 1), (520, 170, 328, 11, 1), (256, 200, 256, 13, 1),
                                                     (264, 416, 72, 13, 1), (512, 230, 512, 15, 1), (256, 480, 192, 15, 1), (512, 205, 640, 13, 3),
                                                     (512, 300, 704, 10, 2), (264, 190, 512, 12, 3), (520, 440, 1088, 14, 5), (256, 65, 512, 8, 8),
                                                     (512, 160, 4104, 10, 4)])
@pytest.mark.parametrize("epilogue", [0, 1, 2])
def test_every_width_whole_and_split(m, n, k, token_tiles, split, epilogue):
    import torch

    from tuna_amd import _lib, ops

    cfg = _cfg(token_tiles, split)
    assert re.match(rf"gemm_wide_kernel<256 rows x \d+ tokens> split_k={split}", ops.describe_launch(m, n, k, cfg))
    q, s, x, code = _inputs(m, n, k, seed=m + n)
    plain, again = _out(n, m), _out(n, m)
    ops.matmul(x, q, s, code, plain, m, n, k, config=cfg)
    ops.matmul(x, q, s, code, again, m, n, k, config=cfg)
    torch.cuda.synchronize()
    assert torch.equal(plain, again)
    _check(plain, q, s, x, code, k)
    if split == 1:  # (the same products in the same order, whatever the width)
        other = _out(n, m)
        ops.matmul(x, q, s, code, other, m, n, k, config=_cfg256(1))
        torch.cuda.synchronize()
        assert torch.equal(plain, other)
    if epilogue:
        res = torch.randn(n * m + 4, device="cuda").half()[4:].view(n, m)  # (aligned to 8 bytes, no more)
        fused = _out(n, m // epilogue)
        ops.matmul_fused(x, q, s, code, fused, m, n, k, epilogue, res if epilogue == _lib.EPILOGUE_RESIDUAL else None, config=cfg)
        torch.cuda.synchronize()
        p = plain.float()
        want = p + res.float() if epilogue == _lib.EPILOGUE_RESIDUAL else torch.nn.functional.silu(p[:, 0::2]) * p[:, 1::2]
        assert (fused.float() - want).abs().max() <= 4e-3 * want.abs().max()


# the last tiles shared between the compute units: segments of any number of steps, one round and whole rounds ahead of it
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,token_tiles,block", [(9728, 620, 4160, 10, 0), (16640, 700, 2112, 12, 0), (8448, 880, 1664, 14, 0), (33024, 1000, 512, 16, 0),
                                                     (9728, 620, 4096, 10, 64), (8448, 1100, 1792, 14, 128), (12800, 500, 2816, 8, 256),
                                                     (9728, 420, 4160, 9, 0), (8448, 860, 1792, 11, 128)])
def test_shared_tiles_of_every_width(m, n, k, token_tiles, block):
    import torch

    from tuna_amd import ops

    cfg = _cfg(token_tiles, 0)
    assert "last tiles shared" in ops.describe_launch(m, n, k, cfg)
    q, s, x, code = _inputs(m, n, k, seed=n, block=block)
    outs = [_out(n, m) for _ in range(3)]
    for o in outs:
        if block:
            ops.matmul_blockwise(x, q, s, code, o, m, n, k, block, config=cfg)
        else:
            ops.matmul(x, q, s, code, o, m, n, k, config=cfg)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    _check(outs[0], q, s, x, code, k, block=block)


# scale blocks: two blocks of a row and more, one step to a block and several, odd numbers of steps, parts that begin inside a block
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,block,token_tiles,split", [(256, 200, 256, 64, 14, 1), (272, 150, 256, 128, 10, 1), (528, 300, 1280, 64, 10, 1),
                                                           (272, 70, 768, 256, 8, 1), (512, 385, 2048, 128, 14, 3), (1024, 129, 1792, 64, 12, 2),
                                                           (512, 180, 2304, 128, 12, 5), (256, 250, 2816, 256, 16, 7), (1280, 768, 5632, 64, 16, 3),
                                                           (512, 140, 2304, 64, 9, 3), (256, 230, 1280, 128, 15, 1)])
def test_scale_blocks_of_every_width(m, n, k, block, token_tiles, split):
    import torch

    from tuna_amd import ops

    q, s, x, code = _inputs(m, n, k, seed=k + n, block=block)
    out = _out(n, m)
    ops.matmul_blockwise(x, q, s, code, out, m, n, k, block, config=_cfg(token_tiles, split))
    torch.cuda.synchronize()
    _check(out, q, s, x, code, k, block=block)


# groups of all widths, whole tiles (one and several rounds), shared ones, a k tail; what lies beyond a group's tokens is the next group's
@pytest.mark.gpu
@pytest.mark.parametrize("m,k,counts", [(2048, 1024, (70, 150, 180, 222, 250, 0, 470, 129)), (8448, 328, (300, 66, 64, 80, 100, 512)),
                                        (1024, 4096, (128, 129, 256, 257)), (4096, 2112, (130, 150, 190, 220, 700, 95, 333, 481)),
                                        (8192, 192, (65, 97, 140, 161, 200, 230, 300))])
def test_groups_of_several_widths(m, k, counts):
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


def test_a_call_without_a_config_takes_the_width_that_is_predicted_to_be_fastest():
    from tuna_amd import ops

    for (m, n, k), tokens in (((4096, 2000, 4096), 128), ((28672, 2000, 4096), 224), ((6144, 2000, 4096), 208)):
        assert ops.describe_launch(m, n, k).startswith(f"gemm_wide_kernel<256 rows x {tokens} tokens>"), (m, n, k)
    c, _hit = ops.select_config_blockwise(4096, 777, 14336, 128)
    assert (c.lds_tile_rows, c.waves_m, c.split_k) == (256, 10, 3)
    assert not ops.describe_launch(4096, 64, 14336).startswith("gemm_wide_kernel")


# (whole tiles; split ones, of which a launch runs an even number of token tiles; shared last tiles)
@pytest.mark.parametrize("m,n,k,token_tiles,split,ends", [(4096, 2000, 4096, 8, 1, "128 tokens> split_k=1 (gemm_wide_whole_kernel)"),
                                                          (7552, 826, 21632, 13, 2, "224 tokens> split_k=2"),
                                                          (10816, 351, 4032, 8, 0, "128 tokens> split_k=1, last tiles shared")])
def test_a_pick_is_described_as_its_config_is(m, n, k, token_tiles, split, ends):
    from tuna_amd import ops

    pick, _, before = ops.describe_launch(m, n, k).partition(" in place of ")
    assert before and pick == ops.describe_launch(m, n, k, _cfg(token_tiles, split))
    assert pick.endswith(ends)


def test_configs_that_no_kernel_runs_are_refused():
    from tuna_amd import _lib, ops

    for token_tiles, split in ((7, 0), (17, 0), (16, -1), (16, 17)):  # (tiles of 256 tokens only are divided into one part and more)
        with pytest.raises(ops.TunaError):
            ops.validate_config(1024, 300, 1024, _cfg(token_tiles, split))
    ops.validate_config(1024, 300, 1024, _cfg(16, 16))
    with pytest.raises(ops.TunaError):
        ops.validate_config(1024, 300, 1024, _cfg(16, 1), _lib.DECODE_DEQUANT)


def test_launches_of_any_number_of_steps_are_planned():
    """Shares are worked out in 32 bits, whole tiles are not: a launch of more steps than that is whole tiles, not refused."""
    from tuna_amd import ops

    for m, n, k in ((57344, 262144, 28672), (57344, 300000, 28672), (131072, 131072, 28672), (152064, 400000, 8192), (40960, 52000, 204800)):
        for cfg in (_cfg256(1), _cfg256(2), _cfg(16, 1), _cfg(16, 2), _cfg(13, 1)):
            ops.validate_config(m, n, k, cfg)
            sums = ops.config_footprint(m, n, k, cfg)[1]  # (256 x 256 tiles, unsplit: the last ones behind whole rounds may be shared)
            assert sums == 0 or (cfg.waves_m, cfg.split_k) == (1, 1) and sums < 1 << 28
            assert ops.describe_launch(m, n, k, cfg).startswith("gemm_wide_kernel")
        assert ops.describe_launch(m, n, k).startswith("gemm_wide_kernel")
    for cfg in (_cfg256(1), _cfg256(3), _cfg(16, 1)):
        ops.validate_config_blockwise(62912, 638681, 30720, 128, cfg)
        ops.validate_config_blockwise(44800, 933118, 29184, 256, cfg)
    # the most steps that are still divided, and one tile more
    tiles, steps = 1024, 0x7fffffff // 21 // 1024
    assert ops.config_footprint(256, 256 * tiles, 64 * steps, _cfg256(3))[1] > 0
    assert ops.config_footprint(256, 256 * (tiles + 1), 64 * steps, _cfg256(3))[1] == 0


def test_an_unsplit_config_of_up_to_half_a_round_of_tiles_needs_no_workspace():
    from tuna_amd import ops

    for m, n, k in ((8832, 497, 3456), (20992, 201, 7680), (2816, 2293, 14784), (17920, 4, 5376), (32768, 256, 28672)):
        assert ops.config_footprint(m, n, k, _cfg256(1))[1] == 0, (m, n, k)
        assert "shared" not in ops.describe_launch(m, n, k, _cfg256(1))


def test_the_static_entry_point_refuses_no_pick_of_many_tokens_for_its_workspace():
    import random

    import torch

    if torch.cuda.is_available():
        pytest.skip("would launch on addresses that are not memory")
    from tuna_amd import _lib

    p, rng = 1 << 20, random.Random(8)
    for _ in range(1500):
        m, n, k = 64 * rng.randrange(16, 800), rng.randrange(65, 3000), 64 * rng.randrange(16, 300)
        assert _lib.lib().tuna_matmul_static(p, p, p, p, p, m, n, k, None, _lib.DECODE_GEMM, None) != _lib.ERR_WORKSPACE, (m, n, k)


@pytest.mark.parametrize("source,kernels", [("gemm_wide.hip", 3), ("gemm_wide_whole.hip", 29)])
def test_no_accumulator_moves_inside_a_loop(tmp_path, source, kernels):
    """The accumulators of the inline assembly MFMAs stay where they are while steps run (a copy the compiler makes there may read one
    that has not been written yet), and nothing touches a register that a load is on its way to."""
    from test_async_loads import CSRC, _follow, _functions

    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    with open(os.path.join(CSRC, "Makefile")) as f:
        flags = re.search(r"^HIPFLAGS \?= ((?:.*\\\n)*.*)", f.read(), re.M).group(1).replace("\\\n", " ").replace("$(ARCH)", "gfx950")
    out = tmp_path / "kernels.s"
    subprocess.run([hipcc, *flags.split(), "--offload-device-only", "-S", source, "-o", str(out)], cwd=CSRC, check=True, capture_output=True)
    found = 0
    for name, body in _functions(out.read_text()):
        loads, early = _follow(body)
        assert not early, (name, early[:4])
        assert not any(t.startswith("scratch_") for t, _ in body), name
        found += loads > 0
        mfma, moved = 0, []  # of the straight-line piece at hand
        for text, _ in body + [("s_branch", False)]:
            mfma += text.startswith("v_mfma")
            moved += [text] if "accvgpr" in text else []
            if text.endswith(":") or text.startswith(("s_cbranch", "s_branch")):
                assert mfma < 2 or not moved, (name, moved[:2])
                mfma, moved = 0, []
    assert found == kernels


@pytest.mark.parametrize("kind,off", [("width", 2.9), ("width blocks", 3.8)])
def test_the_stated_errors_are_those_of_the_kept_launches(kind, off):
    """(per cent, as stated beside width_time in csrc/api.cpp)"""
    from test_launch_models import DATA
    from tuna_amd import launch_models as lm

    rows = [r for r in lm.read(DATA) if r["kind"] == kind]
    assert len(rows) == 440
    assert 100 * lm.errors(rows, *lm.MODELS[kind])[0] == pytest.approx(off, abs=0.06)
