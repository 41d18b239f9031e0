"""Launches without a config where the library's first pick has no room for its partial sums: through the fixed scratch of
tuna_matmul_static, and on a capturing stream whose workspace cannot grow.  The call then runs another launch."""
import random

import numpy as np
import pytest

from helpers import launched
from test_wide_tile import _check, _inputs, _out
from tuna_amd import _lib, ops


def _status_static(m, n, k):
    """Status of tuna_matmul_static up to the point where it needs a device (the pointers are never read)."""
    p = 1 << 20
    return _lib.lib().tuna_matmul_static(p, p, p, p, p, m, n, k, None, _lib.DECODE_GEMM, None)


def test_the_static_entry_point_refuses_no_pick_of_the_library_for_its_workspace():
    import torch

    if torch.cuda.is_available():
        pytest.skip("would launch on addresses that are not memory")
    rng = random.Random(4)
    shapes = [(28672, 37, 8192), (22016, 33, 4096), (27648, 40, 5120), (57344, 48, 8192)]
    shapes += [(64 * rng.randrange(4, 900), rng.randrange(17, 65), 64 * rng.randrange(16, 400)) for _ in range(1500)]
    refused = [s for s in shapes if _status_static(*s) == _lib.ERR_WORKSPACE]
    assert not refused, refused[:5]


# (kernel, m, n, k) whose partial sums fit the static scratch: decode-batch shares that cross tiles and equal parts of tiles, tall
# and broad tiles in parts of k
SHARED = [("gemm_flow_kernel", 33352, 24, 1088), ("gemm_flow_kernel", 33832, 16, 6336), ("gemm_flow_kernel", 33056, 35, 1024),
          ("gemm_tall_kernel", 4096, 64, 14336), ("gemm_tall_kernel", 5120, 37, 13824), ("gemm_broad_kernel", 8192, 160, 8192)]
# ... and whole tiles
WHOLE = [("gemm_tall_kernel", *s) for s in ((22016, 33, 4096), (27648, 40, 5120), (17024, 24, 1936), (17728, 50, 4096), (17664, 14, 5056))]


def test_these_launches_are_what_they_are_here_for():
    for kernel, *shape in SHARED + WHOLE:
        ran, sums = launched(*shape)
        assert ran == kernel and (0 < sums <= 16 << 20 if (kernel, *shape) in SHARED else sums == 0), (shape, ran, sums)


@pytest.mark.gpu
@pytest.mark.parametrize("kernel,m,n,k", SHARED + WHOLE)
def test_static_entry_point(kernel, m, n, k):
    import torch

    assert launched(m, n, k)[0] == kernel
    q, s, x, code = _inputs(m, n, k, seed=n)
    out, again, grown = (_out(n, m) for _ in range(3))
    ops.matmul_static(x, q, s, code, out, m, n, k)
    ops.matmul_static(x, q, s, code, again, m, n, k)
    ops.matmul(x, q, s, code, grown, m, n, k)
    torch.cuda.synchronize()
    assert torch.equal(out, again) and torch.equal(out, grown)  # (the same launch: its sums fit both workspaces)
    _check(out, q, s, x, code, k)


def _calls():
    """(name, bytes of partial sums of an eager call, call, output, check, whether there is a launch without partial sums)"""
    for _kernel, m, n, k in SHARED + [("gemm_flow_kernel", 33136, 41, 1088), ("gemm_wide_kernel", 10816, 351, 4032)]:
        q, s, x, code = _inputs(m, n, k, seed=n)
        out = _out(n, m)
        yield (f"matmul {m} {n} {k}", launched(m, n, k)[1], lambda q=q, s=s, x=x, code=code, out=out, m=m, n=n, k=k:
               ops.matmul(x, q, s, code, out, m, n, k), out, lambda q=q, s=s, x=x, code=code, out=out, k=k: _check(out, q, s, x, code, k),
               ops.config_footprint(m, n, k, ops.select_config(m, n, k)[0])[1] == 0 or _kernel == "gemm_wide_kernel")
    # (scale blocks: 256 x 256 tiles split in parts, tall tiles and broad tiles in parts of k)
    for tile_rows, m, n, k, block in ((256, 8832, 467, 3328, 64), (-6, 4096, 32, 14336, 128), (-6, 4096, 48, 14336, 64), (-7, 4096, 160, 14336, 128)):
        cfg, _hit = ops.select_config_blockwise(m, n, k, block)
        q, s, x, code = _inputs(m, n, k, seed=n, block=block)
        out = _out(n, m)
        yield (f"matmul_blockwise {m} {n} {k}", ops.config_footprint(m, n, k, cfg)[1] if cfg.lds_tile_rows == tile_rows else 0,
               lambda q=q, s=s, x=x, code=code, out=out, m=m, n=n, k=k, block=block: ops.matmul_blockwise(x, q, s, code, out, m, n, k, block),
               out, lambda q=q, s=s, x=x, code=code, out=out, k=k, block=block: _check(out, q, s, x, code, k, block=block), tile_rows != -7)


@pytest.mark.gpu
@pytest.mark.parametrize("warm", [False, True])
def test_capture(warm):
    """Cold: nothing has run on the capturing stream, which has no workspace - other kernels, within the GEMM's tolerance.
    Warm: the shape ran there once, and the graph replays the bits of that run."""
    import torch

    for name, sums, call, out, check, runs_without in _calls():
        print(name, "warm" if warm else "cold", sums, flush=True)
        assert sums > 0
        if not warm and not runs_without:  # (what the pick stands in for splits k itself: such a call asks for the workspace)
            continue
        torch.cuda.synchronize()
        assert _lib.lib().tuna_release_workspaces() == _lib.OK
        side, g, eager = torch.cuda.Stream(), torch.cuda.CUDAGraph(), None
        if warm:
            with torch.cuda.stream(side):
                call()
            side.synchronize()
            eager = out.clone()
        with torch.cuda.graph(g, stream=side):
            call()
        for _ in range(3):
            out.fill_(float("nan"))
            g.replay()
            torch.cuda.synchronize()
            check()
            if warm:
                assert torch.equal(out, eager)
            assert np.isfinite(out.float().sum().item())  # (work of the program between the replays)
    assert _lib.lib().tuna_release_workspaces() == _lib.OK
