"""Launches whose tiles are shared between workgroups, on two streams at once: each stream has partial sums and counters of
its own, and the bits are those of a launch alone."""
import pytest

from test_wide_tile import _check, _inputs, _out

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel,m,n,k", [("gemm_flow_kernel", 22016, 33, 4096), ("gemm_flow_kernel", 17664, 14, 5056),
                                          ("last tiles shared", 8448, 1100, 4096), ("split_k=3 in place", 8832, 497, 3456)])
def test_two_streams(kernel, m, n, k):
    import torch

    from tuna_amd import ops

    assert kernel in ops.describe_launch(m, n, k)
    calls = [_inputs(m, n, k, seed=seed) for seed in (n, n + 1)]
    alone = [_out(n, m) for _ in calls]
    for (q, s, x, code), out in zip(calls, alone):
        ops.matmul(x, q, s, code, out, m, n, k)
        torch.cuda.synchronize()
        _check(out, q, s, x, code, k)
    streams = [torch.cuda.Stream() for _ in calls]
    outs = [[_out(n, m) for _ in range(4)] for _ in calls]
    torch.cuda.synchronize()
    for i in range(4):
        for (q, s, x, code), stream, out in zip(calls, streams, outs):
            with torch.cuda.stream(stream):
                ops.matmul(x, q, s, code, out[i], m, n, k)
    torch.cuda.synchronize()
    for want, out in zip(alone, outs):
        for o in out:
            assert torch.equal(o, want)


@pytest.mark.parametrize("m,k,counts", [(14336, 1024, (3, 0, 17, 33, 1, 16, 8, 2)), (4096, 1024, (400, 100, 777, 90))])
def test_groups_on_two_streams(m, k, counts):
    import numpy as np
    import torch

    from tuna_amd import ops

    offs = np.concatenate([[0], np.cumsum(counts)]).tolist()
    calls = [_inputs(m * len(counts), offs[-1], k, seed=seed) for seed in (k, k + 1)]
    alone = [_out(offs[-1], m) for _ in calls]
    for (q, s, x, code), out in zip(calls, alone):
        ops.matmul_grouped(x, q, s, code, out, m, len(counts), k, offs)
        torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in calls]
    outs = [[_out(offs[-1], m) for _ in range(4)] for _ in calls]
    torch.cuda.synchronize()
    for i in range(4):
        for (q, s, x, code), stream, out in zip(calls, streams, outs):
            with torch.cuda.stream(stream):
                ops.matmul_grouped(x, q, s, code, out[i], m, len(counts), k, offs)
    torch.cuda.synchronize()
    for want, out in zip(alone, outs):
        for o in out:
            assert torch.equal(o, want)
