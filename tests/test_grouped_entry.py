"""Grouped launches without a config: a table entry for the active rows comes before the decode-batch kernel."""
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("m,k,tokens", [(28672, 4096, 1), (28672, 4096, 4), (28672, 4096, 16)])
def test_the_tables_entry_for_the_active_rows_is_what_runs(m, k, tokens):
    """The bits of the call with that entry as its config (the decode-batch kernel sums in another order)."""
    import torch

    from test_wide_tile import _check, _inputs, _out
    from tuna_amd import ops

    groups = 8
    offs = [tokens * e for e in range(groups + 1)]
    assert ops.select_config(m * groups, tokens, k)[1]
    cfg = ops.select_config_grouped(m, groups, tokens, k)
    q, s, x, code = _inputs(m * groups, offs[-1], k, seed=tokens)
    out, named = _out(offs[-1], m), _out(offs[-1], m)
    ops.matmul_grouped(x, q, s, code, out, m, groups, k, offs)
    ops.matmul_grouped(x, q, s, code, named, m, groups, k, offs, config=cfg)
    torch.cuda.synchronize()
    assert torch.equal(out, named)
    for e in (0, 5):
        lo, hi = offs[e], offs[e + 1]
        _check(out[lo:hi], q, s, x[lo:hi], code, k, first_row=e * m, rows=m)
