"""The 256 x 256 many-token tile (csrc/gemm_wide.hip): tiles whole, split, and shared between workgroups; groups in one
launch; scale blocks.  Whole outputs against float64 sums, a subset of rows against the oracle, and deterministic."""
import numpy as np
import pytest

from helpers import O, REL_FLOOR, REL_TOL, f16_bits_to_f64, rel_err

pytestmark = pytest.mark.gpu


def _inputs(m, n, k, seed, block=0):
    import torch

    from tuna_amd.quantize import nf4_codebook
    from tuna_amd.synth import make_weights_torch, make_x_torch

    dev = torch.device("cuda")
    q, s = make_weights_torch(m, k, seed=seed, device=dev)
    if block:
        g = torch.Generator(device=dev)
        g.manual_seed(seed)
        s = torch.empty((m, k // block), device=dev).uniform_(0.005, 0.02, generator=g)
    return q, s, make_x_torch(n, k, seed=seed + 1, device=dev), nf4_codebook(dev)


def _out(n, m):
    import torch

    return torch.full((n, m), float("nan"), dtype=torch.float16, device="cuda")


def _f64_sums(q, s, x, code, k, block):
    """x @ decode(q, code, s)^T in float64 (weights: an fp16 code times an fp16 scale, rounded to fp16), in plain torch."""
    import torch

    nib = torch.stack((q >> 4, q & 15), dim=-1).view(-1, k // 8, 8, 8)          # block row, block column, row, column
    nib = nib.permute(0, 2, 1, 3).reshape(-1, k).long()
    scale = s.half().view(nib.shape[0], -1).repeat_interleave(block or k, dim=1)
    return x.double() @ (code.half()[nib] * scale).double().t().contiguous()


def _check(out, q, s, x, code, k, blocks=6, block=0, first_row=0, rows=None):
    """All of out against float64 sums in torch; rows of `blocks` random block rows (and the last one) against the oracle's,
    whose decode is another implementation."""
    import torch

    m = rows or out.shape[1]
    assert not torch.isnan(out).any()
    own = slice(first_row, first_row + m)
    sums = _f64_sums(q[first_row // 8:(first_row + m) // 8], s[own], x, code, k, block)
    den = sums.abs().clamp_min(REL_FLOOR * float(sums.abs().max()))
    assert float(((out.double() - sums).abs() / den).max()) <= REL_TOL
    rng = np.random.default_rng(m + out.shape[0])
    mbs = np.unique(np.append(rng.choice(m // 8, size=min(blocks, m // 8), replace=False), m // 8 - 1))
    rs = (mbs[:, None] * 8 + np.arange(8)[None, :]).ravel()
    q_sub = q[torch.from_numpy(mbs + first_row // 8).cuda()].cpu().numpy()
    s_sub = s[torch.from_numpy(rs + first_row).cuda()].cpu().numpy()
    xb, cb = x.cpu().numpy().view(np.uint16), code.cpu().numpy()
    ref = O.gemm_f64(q_sub, xb, cb, s_sub, len(rs), x.shape[0], k, mode=O.D1, block_size=block or None)
    got = out.cpu().numpy().view(np.uint16)[:, rs]
    assert rel_err(f16_bits_to_f64(got), ref) <= REL_TOL


def _cfg(split):
    from tuna_amd.ops import GemmConfig

    return GemmConfig.from_dict(dict(rows_per_wave=64, waves_m=1, waves_k=1, split_k=split, prefetch=2, x_chunk=64, token_tiles=16,
                                     xcd_swizzle=0, lds_tile_rows=256))


# whole tiles: 1 .. 128 tokens in the last tile, 129 .. 256, ragged rows; splits with two and more contributors, parts of
# one step, an odd number of steps; k tails
@pytest.mark.parametrize("m,n,k,split", [(256, 128, 128, 1), (264, 129, 64, 1), (520, 384, 192, 1), (1024, 257, 320, 2),
                                         (512, 385, 704, 3), (264, 640, 1088, 5), (256, 100, 512, 8), (512, 129, 1000, 2),
                                         (768, 300, 4104, 7)])
@pytest.mark.parametrize("epilogue", [0, 1, 2])
def test_whole_and_split_tiles(m, n, k, split, epilogue):
    import torch

    from tuna_amd import _lib, ops

    q, s, x, code = _inputs(m, n, k, seed=m + n)
    plain, again = _out(n, m), _out(n, m)
    ops.matmul(x, q, s, code, plain, m, n, k, config=_cfg(split))
    ops.matmul(x, q, s, code, again, m, n, k, config=_cfg(split))
    torch.cuda.synchronize()
    assert torch.equal(plain, again)
    _check(plain, q, s, x, code, k)
    if epilogue:
        res = torch.randn(n, m, device="cuda").half()
        fused = _out(n, m // epilogue)
        ops.matmul_fused(x, q, s, code, fused, m, n, k, epilogue, res if epilogue == _lib.EPILOGUE_RESIDUAL else None, config=_cfg(split))
        torch.cuda.synchronize()
        p = plain.float()
        want = p + res.float() if epilogue == _lib.EPILOGUE_RESIDUAL else torch.nn.functional.silu(p[:, 0::2]) * p[:, 1::2]
        assert (fused.float() - want).abs().max() <= 4e-3 * want.abs().max()


# one round of shares (two and three contributors to a tile), one round of whole tiles and shares, with small last tiles
@pytest.mark.parametrize("m,n,k", [(9728, 1000, 8256), (8448, 1100, 4096), (10240, 2000, 4096)])
def test_last_tiles_shared_between_the_compute_units(m, n, k):
    import torch

    from tuna_amd import ops

    assert "last tiles shared" in ops.describe_launch(m, n, k, _cfg(1))
    q, s, x, code = _inputs(m, n, k, seed=n)
    outs = [_out(n, m) for _ in range(3)]
    for o in outs:
        ops.matmul(x, q, s, code, o, m, n, k, config=_cfg(1))
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    _check(outs[0], q, s, x, code, k)


def test_a_capturing_stream_without_workspace_takes_whole_tiles():
    """Sharing needs room for partial sums, which cannot be allocated during a capture: the launch then runs whole tiles."""
    import torch

    from tuna_amd import ops

    m, n, k = 9728, 1000, 8256
    q, s, x, code = _inputs(m, n, k, seed=5)
    shared, out = _out(n, m), _out(n, m)
    ops.matmul(x, q, s, code, shared, m, n, k, config=_cfg(1))
    torch.cuda.synchronize()
    g, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(g, stream=side):
        ops.matmul(x, q, s, code, out, m, n, k, config=_cfg(1))
    for _ in range(3):
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert (out.float() - shared.float()).abs().max() <= 2e-3 * shared.float().abs().max()


@pytest.mark.parametrize("m,k,counts", [(512, 512, (200, 65, 0, 128, 129, 256, 257, 70)), (320, 1032, (300, 66, 64, 80, 100, 512)),
                                        (2048, 1024, (400, 1, 777, 90)), (4608, 2688, (5, 1250, 0, 420, 30))])
def test_groups_of_many_tokens_in_one_launch(m, k, counts):
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


# scale blocks: one block per step and several steps per block, odd numbers of steps, splits, small last tiles
@pytest.mark.parametrize("m,n,k,block,split", [(256, 200, 256, 64, 1), (528, 300, 1280, 64, 1), (272, 70, 768, 256, 1), (512, 385, 2048, 128, 3),
                                               (1024, 129, 1792, 64, 2), (1280, 768, 5632, 64, 3)])
def test_scale_blocks(m, n, k, block, split):
    import torch

    from tuna_amd import ops

    q, s, x, code = _inputs(m, n, k, seed=k + n, block=block)
    out = _out(n, m)
    ops.matmul_blockwise(x, q, s, code, out, m, n, k, block, config=_cfg(split))
    torch.cuda.synchronize()
    _check(out, q, s, x, code, k, block=block)


# the same in launches whose last tiles are shared: segments of any number of steps, full token tiles and small last ones
@pytest.mark.parametrize("m,n,k,block", [(9728, 1024, 8192, 64), (8448, 1100, 4352, 128), (5120, 2000, 13824, 64)])
def test_scale_blocks_of_shared_tiles(m, n, k, block):
    import torch

    from tuna_amd import ops

    assert "last tiles shared" in ops.describe_launch(m, n, k, _cfg(1))
    q, s, x, code = _inputs(m, n, k, seed=k + n, block=block)
    outs = [_out(n, m) for _ in range(3)]
    for o in outs:
        ops.matmul_blockwise(x, q, s, code, o, m, n, k, block, config=_cfg(1))
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    _check(outs[0], q, s, x, code, k, block=block)
