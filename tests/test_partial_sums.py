"""Room for partial sums of the kernels whose k-steps are divided into shares: two slots per share only where a share can have
parts of two tiles, one where every tile ends with a share, none where no tile is divided."""
import pytest

from tuna_amd import ops

SLOT_WIDE = 256 * 256 * 4 + 4352


def _flow(n, shares):
    return ops.GemmConfig.from_dict(dict(rows_per_wave=64, waves_m=4, waves_k=1, split_k=shares, prefetch=4, x_chunk=64,
                                         token_tiles=-(-n // 16), xcd_swizzle=0, lds_tile_rows=-4))


def _wide(split):
    return ops.GemmConfig.from_dict(dict(rows_per_wave=64, waves_m=1, waves_k=1, split_k=split, prefetch=2, x_chunk=64, token_tiles=16,
                                         xcd_swizzle=0, lds_tile_rows=256))


def _most_parts(steps, shares):
    """Largest number of divided tiles that one share has parts of (steps: the work of each tile)."""
    ends = [0]
    for s in steps:
        ends.append(ends[-1] + s)
    most = 0
    for i in range(shares):
        lo, hi = ends[-1] * i // shares, ends[-1] * (i + 1) // shares
        most = max(most, sum(lo < e and hi > b and not (lo <= b and e <= hi) for b, e in zip(ends, ends[1:])))
    return most


@pytest.mark.parametrize("m,n,k,shares", [(256, 1, 64, 1), (512, 17, 1024, 2), (1024, 48, 4096, 2), (776, 33, 4096, 7), (1024, 48, 1288, 16),
                                          (2048, 49, 2048, 5), (256, 64, 4104, 16), (8192, 16, 4096, 512), (28672, 37, 8192, 224),
                                          (28672, 37, 8192, 512), (4096, 5, 1000, 64), (1024, 8, 64, 512)])
def test_decode_batch_kernel(m, n, k, shares):
    tiles, units = -(-m // 256), -(-(-(-k // 64)) // 4)
    shares_run = min(shares, tiles * units)
    slots = _most_parts([units] * tiles, shares_run)
    got = ops.config_footprint(m, n, k, _flow(n, shares))[1]
    assert got == shares_run * slots * 256 * 16 * -(-n // 16) * 4


@pytest.mark.parametrize("m,n,k,split,slots", [(512, 512, 4096, 1, 0), (512, 512, 4096, 3, 1), (256, 100, 512, 2, 1), (512, 640, 4096, 4, 2),
                                               (4096, 777, 14336, 4, 2), (4096, 768, 14336, 4, 1)])
def test_256_x_256_tile(m, n, k, split, slots):
    tiles = -(-m // 256) * -(-n // 256)
    assert ops.config_footprint(m, n, k, _wide(split))[1] == (tiles * split if split > 1 else 0) * slots * SLOT_WIDE
