"""The weight loads of the 256-row kernels at the edges of the matrix: their offsets, checked on the host for what a buffer
descriptor's range check accepts, and the launches at the shapes where an offset could leave the weights."""
import ctypes

import pytest

from tuna_amd import _lib

# 8 rows in the last row tile and 8, 16 or 24 k values in the last step: a step's uniform offset could exceed the buffer
EDGES = [(8, 8), (8, 72), (264, 72), (264, 80), (264, 88), (520, 1048), (264, 4104)]


@pytest.mark.parametrize("kernel", [0, 1])
def test_no_accepted_load_reaches_behind_the_weights(kernel):
    L = _lib.bench_lib()
    out = (ctypes.c_longlong * 4)()
    for m in (8, 16, 24, 64, 136, 248, 256, 264, 272, 520):
        for k in [8 * i for i in range(1, 18)] + [504, 512, 1000, 1024, 1032, 1040, 1048, 4104]:
            for tile in range(-(-m // 256)):
                assert L.tuna_check_weight_reach(kernel, m, k, tile, out) == _lib.OK
                assert list(out) == [0, 0, 0, 0], (m, k, tile)


@pytest.mark.gpu
@pytest.mark.parametrize("m,k", EDGES)
def test_launches_at_the_edges(m, k):
    import torch

    from test_flow_kernel import _cfg as flow
    from test_wide_tile import _cfg as wide, _check, _inputs, _out
    from tuna_amd import ops

    for n, cfg in ((5, flow(5, 1)), (40, flow(40, 2)), (5, wide(1)), (200, wide(1))):
        q, s, x, code = _inputs(m, n, k, seed=m + k)
        out = _out(n, m)
        ops.matmul(x, q, s, code, out, m, n, k, config=cfg)
        torch.cuda.synchronize()
        _check(out, q, s, x, code, k)
