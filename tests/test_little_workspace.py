"""Launches without a config where the library's first pick has no room for its partial sums: through the fixed scratch of
tuna_matmul_static.  The call then runs another launch."""
import random

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
