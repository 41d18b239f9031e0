"""Launches without a config where the library's first pick has no room for its partial sums: through the fixed scratch of
tuna_matmul_static, and on a capturing stream whose workspace cannot grow.  The call then runs another launch."""
import random

import numpy as np
import pytest

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


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(22016, 33, 4096), (27648, 40, 5120), (17024, 24, 1936), (17728, 50, 4096), (17664, 14, 5056)])
def test_static_entry_point(m, n, k):
    import torch

    assert "gemm_flow_kernel" in ops.describe_launch(m, n, k)
    q, s, x, code = _inputs(m, n, k, seed=n)
    out, again = _out(n, m), _out(n, m)
    ops.matmul_static(x, q, s, code, out, m, n, k)
    ops.matmul_static(x, q, s, code, again, m, n, k)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    _check(out, q, s, x, code, k)


def _calls():
    """(name, kernel that an eager call takes, call, output, check)"""
    for m, n, k in ((22016, 33, 4096), (17024, 24, 1936), (17664, 14, 5056), (8832, 497, 3456)):
        q, s, x, code = _inputs(m, n, k, seed=n)
        out = _out(n, m)
        yield (f"matmul {m} {n} {k}", ops.describe_launch(m, n, k), lambda q=q, s=s, x=x, code=code, out=out, m=m, n=n, k=k:
               ops.matmul(x, q, s, code, out, m, n, k), out, lambda q=q, s=s, x=x, code=code, out=out, k=k: _check(out, q, s, x, code, k))
    m, n, k, block = 8832, 467, 3328, 64
    cfg, _hit = ops.select_config_blockwise(m, n, k, block)
    q, s, x, code = _inputs(m, n, k, seed=n, block=block)
    out = _out(n, m)
    yield (f"matmul_blockwise {m} {n} {k}", f"gemm_wide_kernel split_k={cfg.split_k}" if cfg.lds_tile_rows == 256 and cfg.split_k > 1 else "",
           lambda: ops.matmul_blockwise(x, q, s, code, out, m, n, k, block), out, lambda: _check(out, q, s, x, code, k, block=block))


@pytest.mark.gpu
@pytest.mark.parametrize("warm", [False, True])
def test_capture(warm):
    """Cold: nothing has run on the capturing stream, which has no workspace - other kernels, within the GEMM's tolerance.
    Warm: the shape ran there once, and the graph replays the bits of that run."""
    import torch

    for name, kernel, call, out, check in _calls():
        print(name, "warm" if warm else "cold", kernel, flush=True)
        assert kernel.startswith(("gemm_flow_kernel", "gemm_wide_kernel"))
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
