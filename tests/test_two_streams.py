"""Launches whose tiles are shared between workgroups, on two streams at once: each stream has partial sums and counters of
its own, and the bits are those of a launch alone."""
import pytest

from helpers import launched
from test_wide_tile import _check, _inputs, _out

pytestmark = pytest.mark.gpu


# decode-batch shares that cross tiles (three and one token tile) and equal parts of tiles; tall and broad tiles in parts of k;
# 256-row tiles with the last ones shared, and split in three
@pytest.mark.parametrize("kernel,m,n,k", [("gemm_flow_kernel", 33136, 41, 1088), ("gemm_flow_kernel", 33832, 16, 6336),
                                          ("gemm_flow_kernel", 33056, 35, 1024), ("gemm_tall_kernel", 4096, 64, 14336),
                                          ("gemm_tall_kernel", 5120, 37, 13824), ("gemm_broad_kernel", 8192, 160, 8192),
                                          ("gemm_wide_kernel", 10816, 351, 4032), ("gemm_wide_kernel", 10112, 406, 6272)])
def test_two_streams(kernel, m, n, k):
    import torch

    from tuna_amd import ops

    ran, sums = launched(m, n, k)
    assert ran == kernel and sums > 0
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


# decode-batch shares that are equal parts of tiles, and that cross them; 256-row tiles of groups, whole with decode-batch shares behind
# them, split in two, and with shared last tiles and decode-batch shares whose partial sums lie behind theirs
@pytest.mark.parametrize("m,k,counts", [(2816, 2048, (3, 0, 17, 32, 1, 16, 8, 2)), (4096, 4096, (3, 0, 17, 32, 1, 16, 8, 2)),
                                        (4608, 2688, (5, 1250, 0, 420, 30)), (5120, 1024, (157, 232, 14, 1207, 1494, 4)),
                                        (2048, 3712, (538, 0, 1544)), (6656, 4096, (503, 16, 1981, 42))])
def test_groups_on_two_streams(m, k, counts):
    import numpy as np
    import torch

    from tuna_amd import _lib, ops

    offs = np.concatenate([[0], np.cumsum(counts)]).tolist()
    calls = [_inputs(m * len(counts), offs[-1], k, seed=seed) for seed in (k, k + 1)]
    alone = [_out(offs[-1], m) for _ in calls]
    for (q, s, x, code), out in zip(calls, alone):
        ops.matmul_grouped(x, q, s, code, out, m, len(counts), k, offs)
        torch.cuda.synchronize()
        for e, (lo, hi) in enumerate(zip(offs, offs[1:])):
            if hi > lo:
                _check(out[lo:hi], q, s, x[lo:hi], code, k, first_row=e * m, rows=m)
    # (all kernels are loaded: a call that has no workspace yet takes memory for nothing else)
    assert _lib.lib().tuna_release_workspaces() == _lib.OK
    free = torch.cuda.mem_get_info()[0]
    q, s, x, code = calls[0]
    ops.matmul_grouped(x, q, s, code, alone[0], m, len(counts), k, offs)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] >= 8 << 20
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


# (k of a few steps: whole tiles of the groups' own widths are ahead of shared ones of 256 tokens, and need no partial sums)
def test_a_call_of_few_and_many_tokens_leaves_the_least_workspace():
    import numpy as np
    import torch

    from tuna_amd import _lib, ops

    m, k, counts = 5120, 1024, (157, 232, 14, 1207, 1494, 4)
    offs = np.concatenate([[0], np.cumsum(counts)]).tolist()
    q, s, x, code = _inputs(m * len(counts), offs[-1], k, seed=k)
    out = _out(offs[-1], m)
    ops.matmul_grouped(x, q, s, code, out, m, len(counts), k, offs)
    torch.cuda.synchronize()
    assert _lib.lib().tuna_release_workspaces() == _lib.OK
    free = torch.cuda.mem_get_info()[0]
    for _ in range(2):
        ops.matmul_grouped(x, q, s, code, out, m, len(counts), k, offs)
        torch.cuda.synchronize()
        assert 8 << 20 <= free - torch.cuda.mem_get_info()[0] <= 16 << 20
