"""The narrow-row kernel's ways to its B fragments (narrow_fragments in csrc/tuna_internal.h): a token's result does not depend on how many
tokens go with it, so the first rows of a call with sixteen are, bit for bit, what calls with fewer tokens give."""
import pytest

from test_wide_tile import _check, _inputs, _out

pytestmark = pytest.mark.gpu


def _cfg(rows, wk, u, any_k):
    from tuna_amd.ops import GemmConfig

    return GemmConfig.from_dict(dict(rows_per_wave=rows, waves_m=0 if rows == 64 else 1, waves_k=wk, split_k=1, prefetch=u,
                                     x_chunk=32 * wk * u, token_tiles=1, xcd_swizzle=0, lds_tile_rows=-5 if any_k else 0))


# every tile height with rings of one, two and four double steps, one turn and several; a scale per row and per block; k that ends inside a
# line, inside its first half and before a wave's first step
@pytest.mark.parametrize("m,k,rows,wk,u,block", [(64, 1024, 16, 8, 4, 0), (96, 1024, 32, 16, 2, 0), (96, 2048, 32, 8, 8, 0), (6144, 4096, 24, 8, 4, 0),
                                                 (48, 512, 24, 8, 2, 0), (128, 3072, 64, 8, 4, 0), (64, 1024, 64, 8, 2, 0), (128, 2048, 32, 8, 4, 64),
                                                 (64, 1024, 16, 8, 4, 64), (128, 1024, 64, 8, 2, 128), (40, 1056, 32, 8, 4, -1), (264, 2008, 64, 4, 4, -1),
                                                 (24, 40, 32, 8, 4, -1), (1000, 72, 16, 16, 4, -1), (144, 768, 64, 8, 4, -256)])
def test_tokens_do_not_depend_on_their_company(m, k, rows, wk, u, block):
    import torch

    from tuna_amd import ops

    cfg, any_k, block = _cfg(rows, wk, u, block < 0), block < 0, abs(block) if abs(block) > 1 else 0
    q, s, x, code = _inputs(m, 16, k, seed=m + k + rows, **({"block": block} if block else {}))
    run = (lambda x_, o, n: ops.matmul_blockwise(x_, q, s, code, o, m, n, k, block, config=cfg)) if block else \
        (lambda x_, o, n: ops.matmul(x_, q, s, code, o, m, n, k, config=cfg))
    whole = _out(16, m)
    run(x, whole, 16)
    torch.cuda.synchronize()
    _check(whole, q, s, x, code, k, **({"block": block} if block else {}))
    for n in (1, 4, 5, 7, 8, 9, 15):
        if not block:
            perm = 1 if n > 8 else 0 if n <= 4 else 2 if rows > 16 and not any_k else 1
            assert f"PERM={perm}" in ops.describe_launch(m, n, k, cfg) and ("any k" in ops.describe_launch(m, n, k, cfg)) == any_k
        xs = torch.cat([x[:n].flatten(), torch.full((4096,), float("nan"), dtype=x.dtype, device="cuda")])[:n * k].view(n, k)
        out = _out(n, m)
        run(xs, out, n)
        torch.cuda.synchronize()
        assert torch.equal(out, whole[:n]), n
