"""The time models behind the choice between kernels (flow_time, narrow_time, tall_time, broad_time, wide_time and width_time of csrc/api.cpp): the launches
they are read off, how far they are from them, and the fit of their coefficients.

    python -m tuna_amd.launch_models --measure times.csv    # on a GPU: random shapes, several launches each
    python -m tuna_amd.launch_models --again wide times.csv # on a GPU: one kind's launches of the file once more
    python -m tuna_amd.launch_models times.csv              # anywhere: the models' errors, and refitted coefficients

A model is a function of a launch and a list of coefficients (below, the forms of api.cpp with its coefficients); the fit
minimises the squared logarithm of predicted over measured time, large errors damped (scipy's least_squares, soft_l1).
profiles/launch_model_times.csv holds the launches of one run.
"""
import argparse
import csv
import math
import random

CUS = 256
FIELDS = ("kind", "m", "n", "k", "block", "rows", "waves_k", "prefetch", "token_tiles", "split", "us")


def _cd(a, b):
    return -(-a // b)


# ---- the models: (launch as a dict, coefficients) -> microseconds ------------------------------------------------------

FLOW = (0.916, 1.0, 1.227, 1.302, 0.485, 0.522, 6.1, 2.7, 0.3)


def flow(r, c):
    tiles, units, nt, shares = _cd(r["m"], 256), _cd(_cd(r["k"], 64), 4), r["token_tiles"], r["split"]
    per_share = _cd(tiles * units, shares) * 4
    two = 0.0 if shares <= CUS else shares / CUS - 1.0
    step = (c[4] + c[5] * min(two, 1.0)) * c[nt - 1]
    contributors = shares / tiles + 1.0
    if tiles * units % shares == 0 and tiles * units // shares % units == 0:
        contributors = 1.0
    elif shares % tiles == 0 and units % (shares // tiles) == 0:
        contributors = shares / tiles
    over = c[7] + (c[8] * nt * (contributors - 2.0) if contributors > 2.0 else 0.0) if contributors > 1.0 else 0.0
    return c[6] + per_share * step + over


# launch, round, step, rows, tokens, both, turn, ring, stream, x, scale_loads, scale_kb
NARROW = (1.73, 1.07, 7.5e-5, 0.00291, 0.00252, 0.00691, 0.423, 0.0261, 0.0750, 0.0504, 0.0, 0.0)
NARROW_BLOCKS = (1.98, 2.14, 3.0e-5, 0.00218, 0.00054, 0.00767, 0.0814, 0.190, 0.0355, 0.0461, 0.0220, 0.0642)


def narrow(r, c):
    m, n, k, rows, wk, u, tt = (r[f] for f in ("m", "n", "k", "rows", "waves_k", "prefetch", "token_tiles"))
    nblk = k // r["block"] if r["block"] else 0
    lw, n_it = _cd(rows, 16), _cd(k, 32 * wk * u) * u
    wgs = _cd(m, rows) * _cd(n, 16 * tt)
    lds = 65536 + wk * lw * tt * 1024
    scales = rows * (nblk + 1) * 4 if nblk else 0
    in_lds = lds + scales <= 160 * 1024
    lds += scales if in_lds else 0
    rounds = _cd(wgs, 2 * CUS if lds <= 80 * 1024 else CUS)
    work = _cd(wgs, CUS) * n_it * wk * (c[2] + c[3] * lw + c[4] * tt + c[5] * lw * tt + (0.0 if in_lds else c[10] * lw))
    chain = rounds * n_it / u * (c[6] + c[7] * u)
    stream = c[8] * 0.5e-6 * m * k
    x_mb = wgs * k * min(n, 16 * tt) * 2e-6
    return (c[0] + (c[1] + (c[11] * 1e-3 * scales if in_lds else 0.0)) * rounds +
            (abs(work) ** 3 + abs(chain) ** 3 + abs(stream) ** 3) ** (1 / 3) + c[9] * x_mb)


WIDE = (0.505, 0.907, 0.604, 12.3, 3.7, 17.0, 2.05, 32.1)


def _wide(large, small, steps, split, c):
    tiles = large + small

    def step_us(workgroups):
        return c[1] + c[2] * min(workgroups, CUS) / CUS

    kind = 1.0 if large > 0 else c[0]
    if split == 1:
        if tiles <= CUS:
            return steps * step_us(large + 0.7 * small) * kind + c[3]
        rounds = _cd(large, CUS)
        rest = max(0, small - (rounds * CUS - large))
        total = rounds + _cd(rest, CUS) * c[0]
        last = CUS if rest > 0 or large % CUS == 0 else large % CUS
        return steps * (step_us(CUS) * (total - 1.0) + step_us(last)) + c[3] * total
    if split > 1:
        return (steps / split * step_us(tiles * split) * kind + c[4]) * _cd(tiles * split, CUS) + c[5] + c[6] * (split - 2)
    work = large + small * c[0]
    rounds = max(0, min(math.floor(work / CUS - 0.25), large // CUS))
    per_tile = CUS / (tiles - rounds * CUS) + 1.0
    return (rounds * (steps * step_us(CUS) + c[3]) + (work - rounds * CUS) / CUS * steps * step_us(CUS) + c[7] +
            c[6] * max(0.0, per_tile - 2))


def wide(r, c):
    m, n, k, split = r["m"], r["n"], r["k"], r["split"]
    large, small, steps = _cd(m, 256) * ((n + 127) >> 8), _cd(m, 256) if 1 <= (n & 255) <= 128 else 0, _cd(k, 64)
    if split == 1 and large + small > CUS / 2 and _wide(large, small, steps, 0, WIDE) < _wide(large, small, steps, 1, WIDE):
        split = 0  # (the launch shares its last tiles by itself; by the coefficients in use, whatever is being fitted)
    return _wide(large, small, steps, split, c)


# launch, round, step, rows, tokens, both, tokens where rows of x start inside a cache line, stream, hand-over, its parts, sums, output,
# KB of a workgroup's scales
TALL = (1.519, 2.036, 0.2405, 0.04922, 0.1367, 0.0191, 0.2187, 0.1662, 2.371, 0.02158, 0.02599, 3.18, 0.0)
TALL_BLOCKS = (2.622, 2.036, 0.2332, 0.05657, 0.1367, 0.0191, 0.2187, 0.1662, 2.371, 0.02158, 0.02599, 3.18, 0.0264)


def tall(r, c):
    m, n, k, split = r["m"], r["n"], r["k"], r["split"]
    rt, nt, steps, nblk = r["rows"] // 16, r["token_tiles"], _cd(k, 64), k // r["block"] if r["block"] else 0
    part = _cd(steps, split)
    parts = _cd(steps, part)
    rounds = _cd(_cd(m, 16 * rt) * parts, CUS)
    work = rounds * _cd(part, 8) * (c[2] + c[3] * rt + (c[6] if k % 64 else c[4]) * nt + c[5] * rt * nt)
    stream = c[7] * (0.5e-6 * m * k + 4e-6 * m * nblk)
    scales = c[12] * 0.0625 * rt * math.ceil(part * 64.0 * nblk / k) if nblk else 0.0
    over = c[8] + c[9] * parts * nt * rt if parts > 1 else 0.0
    return c[0] + rounds * (c[1] + c[10] * rt * nt + scales) + (abs(work) ** 3 + abs(stream) ** 3) ** (1 / 3) + over + c[11] * 1e-6 * n * m


# launch, round, unit, rows, tokens, both, tokens where rows of x start inside a cache line, with every compute unit at work,
# hand-over, its parts, sums, output; with scales in blocks launch, round, unit, rows and KB of scales where LDS holds a part's,
# then the first four where it holds a unit's
BROAD = (3.015, 1.578, 0.1557, 0.13, 0.0865, 0.00105, 0.1034, 0.0496, 1.831, 0.0343, 0.0809, 0.8826)
BROAD_BLOCKS = BROAD + (2.484, 3.578, 0.0761, 0.1482, 0.0332, 1.212, 2.125, 0.3803, 0.1493)


def _broad_scales_fit(rt, nt, part, parts, block):
    steps, size = 4 * part, block // 64
    blocks = _cd(steps, size) + (1 if parts > 1 and steps % size else 0)
    return 65536 + 16384 * nt + blocks * 128 * (1 if rt <= 2 else 2 if rt <= 4 else 4) <= 160 * 1024


def broad(r, c):
    m, n, k, nt, split = r["m"], r["n"], r["k"], r["token_tiles"], r["split"]
    rt, units, nblk = r["rows"] // 32, _cd(_cd(k, 64), 4), k // r["block"] if r["block"] else 0
    part = _cd(units, split)
    parts = _cd(units, part)
    own, kb = c[:4], 0.0
    if nblk:
        in_lds = nblk >= 4 and _broad_scales_fit(rt, nt, part, parts, r["block"])
        own, kb = (c[12:16], c[16]) if in_lds else (c[17:21], 0.0)
    full, rest = divmod(_cd(m, r["rows"]) * _cd(n, 16 * nt) * parts, CUS)
    unit = own[2] + own[3] * rt + (c[6] if k % 64 else c[4]) * nt + c[5] * rt * nt
    work = part * (full * (unit + c[7] * nt) + (unit + c[7] * nt * rest / CUS if rest else 0.0))
    scales = kb * 0.125 * rt * math.ceil(part * 256.0 * nblk / k) if nblk else 0.0
    over = c[8] + c[9] * parts * nt * rt if parts > 1 else 0.0
    return own[0] + (full + (1 if rest else 0)) * (own[1] + c[10] * rt * nt + scales) + work + over + c[11] * 1e-6 * n * m


# a k-step's decode, its token tiles, those with every compute unit at work, a tile's end, hand-over, its parts, its sums, where shares
# cross tiles: the ends, the steps
WIDTH = (0.3629, 0.04097, 0.02435, 0.5872, 7.453, 0.1832, 0.5656, 0.4398, 1.058)
WIDTH_BLOCKS = (0.4656, 0.04306, 0.02143, 0.431, 7.898, 0.2, 0.6377, 0.557, 1.034)


def width_tiles(n, token_tiles):
    """Tiles that n tokens make at up to 16 * token_tiles each, and the token tiles of 16 that one runs."""
    count = _cd(n, 16 * token_tiles)
    tokens = _cd(_cd(n, count), 16) * 16
    return count, max(8, tokens // 16)


def kinds_time(kinds, steps, split, c):
    """Tiles of several kinds, (number, token tiles of 16), the widest first."""
    if split != 1:  # (the kernel that divides tiles runs even numbers)
        kinds = [(t, nt + nt % 2) for t, nt in kinds]
    tiles, widest, several = sum(t for t, _ in kinds), kinds[0][1], len(kinds) > 1

    def busy(workgroups):  # share of the compute units at work, over all rounds
        return workgroups / (_cd(workgroups, CUS) * CUS)

    def step(nt, u):
        return c[0] + nt * (c[1] + c[2] * u * u)

    def over(parts, workgroups):
        return c[4] + c[5] * widest * max(0, parts - 2) + c[6] * widest * min(workgroups, CUS) / CUS

    if split == 1:
        # in rounds of a tile per compute unit, each as long as its widest tile
        us, first, seen = 0.0, 0, 0
        for t, nt in kinds:
            seen += t
            rounds = max(0, _cd(seen - first, CUS))
            us, first = us + rounds * (steps * step(nt, busy(tiles)) + c[3] * nt), first + rounds * CUS
        return us
    if split > 1:
        wgs = tiles * split
        work = sum(t * (steps * step(nt, busy(wgs)) / split + c[3] * nt) for t, nt in kinds)
        if several:
            return 1.09 * (_cd(wgs, CUS) * work / tiles * c[8] + c[3] * widest * c[7] + over(split + 1, wgs))
        return _cd(wgs, CUS) * work / tiles + over(split, wgs)
    # as many rounds of whole tiles as wide_balance of csrc/tuna_internal.h leaves, the others shared
    weight, own = sum(t * (nt + 5) * steps for t, nt in kinds), widest + 5
    rounds, shares = min(int(weight / (own * steps * CUS) - 0.25), kinds[0][0] // CUS), CUS
    if not rounds:
        shares = min(shares, 8 * tiles)
        if shares > weight // (8 * own):
            shares = weight // (8 * own) + 1
    whole = rounds * CUS
    us = rounds * (steps * step(widest, 1.0) + c[3] * widest)
    if tiles <= whole:
        return us
    divided = tiles - whole
    ragged = several or (shares % divided and divided % shares)
    work = sum((t - (0 if i else whole)) * steps * step(nt, shares / CUS) for i, (t, nt) in enumerate(kinds))
    us += work / shares * (c[8] if ragged else 1.0) + c[3] * widest * (1.0 + c[7] if ragged else 1.0)
    if several:
        return 1.03 * (us + over(shares / divided + 1.0, shares))
    return us + over(shares / divided + (1.0 if ragged else 0.0), shares) if divided % shares else us


def width(r, c):
    count, nt = width_tiles(r["n"], r["token_tiles"])
    return kinds_time([(_cd(r["m"], 256) * count, nt)], _cd(r["k"], 64), r["split"], c)


MODELS = {"flow": (flow, FLOW), "narrow": (narrow, NARROW), "narrow blocks": (narrow, NARROW_BLOCKS), "wide": (wide, WIDE),
          "tall": (tall, TALL), "tall blocks": (tall, TALL_BLOCKS), "broad": (broad, BROAD), "broad blocks": (broad, BROAD_BLOCKS),
          "width": (width, WIDTH), "width blocks": (width, WIDTH_BLOCKS)}


def config_of(r):
    """The tuna_gemm_config of a launch."""
    from .ops import GemmConfig

    if r["kind"] == "flow":
        d = dict(rows_per_wave=64, waves_m=4, waves_k=1, split_k=r["split"], prefetch=4, x_chunk=64, lds_tile_rows=-4)
    elif r["kind"] in ("tall", "tall blocks"):
        d = dict(rows_per_wave=r["rows"], waves_m=1, waves_k=8, split_k=r["split"], prefetch=2, x_chunk=64, lds_tile_rows=-6)
    elif r["kind"] in ("broad", "broad blocks"):
        d = dict(rows_per_wave=r["rows"], waves_m=2, waves_k=4, split_k=r["split"], prefetch=2, x_chunk=256, lds_tile_rows=-7)
    elif r["kind"] in ("width", "width blocks"):
        d = dict(rows_per_wave=64, waves_m=r["token_tiles"], waves_k=1, split_k=r["split"], prefetch=2, x_chunk=64, lds_tile_rows=256)
        return GemmConfig.from_dict(dict(d, token_tiles=16, xcd_swizzle=0))
    elif r["kind"] == "wide":
        d = dict(rows_per_wave=64, waves_m=1, waves_k=1, split_k=r["split"], prefetch=2, x_chunk=64, lds_tile_rows=256)
    else:
        d = dict(rows_per_wave=r["rows"], waves_m=0 if r["rows"] == 64 else 1, waves_k=r["waves_k"], split_k=1, prefetch=r["prefetch"],
                 x_chunk=32 * r["waves_k"] * r["prefetch"], lds_tile_rows=-5)
    return GemmConfig.from_dict(dict(d, token_tiles=r["token_tiles"], xcd_swizzle=0))


# ---- launches to read them off ---------------------------------------------------------------------------------------

# (rows, waves along k, ring, token tiles): the variants best_narrow_any chooses among
VARIANTS = ((16, 16, 4, 1), (16, 16, 2, 1), (32, 8, 4, 1), (32, 8, 8, 1), (64, 4, 4, 1), (64, 8, 4, 1), (32, 8, 2, 2), (32, 8, 4, 2),
            (64, 8, 2, 2), (32, 8, 2, 4), (64, 4, 2, 4))


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def launches(kind, rng, per_shape):
    """Launches of one random shape."""
    def row(m, n, k, block=0, rows=0, waves_k=0, prefetch=0, token_tiles=0, split=0):
        return dict(kind=kind, m=m, n=n, k=k, block=block, rows=rows, waves_k=waves_k, prefetch=prefetch, token_tiles=token_tiles, split=split)

    if kind == "wide":
        while True:
            m, n, k = 64 * round(_log_uniform(rng, 16, 896)), round(_log_uniform(rng, 65, 4096)), 64 * round(_log_uniform(rng, 16, 400))
            if 2.0 * m * n * k <= 8e11:
                break
        tiles = _cd(m, 256) * _cd(n, 256)
        splits = [s for s in (1, 2, 3, 4, 6, 8) if s == 1 or (tiles * s <= 400 and _cd(k, 64) / s >= 8)]
        return [row(m, n, k, token_tiles=16, split=s) for s in rng.sample(splits, min(per_shape, len(splits)))]
    if kind in ("width", "width blocks"):
        block = rng.choice((64, 128)) if kind == "width blocks" else 0
        while True:
            m, n = 64 * round(_log_uniform(rng, 16, 896)), round(_log_uniform(rng, 65, 4096))
            k = 256 * round(_log_uniform(rng, 4, 112)) if block else 64 * round(_log_uniform(rng, 16, 448))
            fit = []
            for nt in range(8, 17):
                count, own = width_tiles(n, nt)
                tiles = _cd(m, 256) * count
                fit += [(nt, s) for s in (0, 1, 2, 3, 4, 6, 8) if own == nt and
                        (tiles > CUS / 2 if s == 0 else tiles >= 24 if s == 1 else tiles * s <= 400 and _cd(k, 64) / s >= 8)]
            if fit and 2.0 * m * n * k <= 6e11:
                return [row(m, n, k, block, token_tiles=nt, split=s) for nt, s in rng.sample(fit, min(per_shape, len(fit)))]
    lo, hi = (6, 390) if kind == "flow" else (0.5, 400) if kind.startswith(("tall", "broad")) else (0.5, 100)
    unit = 256 if kind.endswith("blocks") else 8
    while True:
        m, k = 16 * round(_log_uniform(rng, 64, 3584)), unit * round(_log_uniform(rng, 1024 / unit, 28672 / unit))
        if lo <= m * k / 2e6 <= hi:
            break
    n = round(_log_uniform(rng, 49, 640) if kind.startswith("broad") else _log_uniform(rng, 1, 64))
    nt = _cd(n, 16)
    if kind == "flow":
        tiles, units = _cd(m, 256), _cd(_cd(k, 64), 4)
        shares = {p * tiles for p in (1, 2, 3, 4, 6, 8)} | {64, 128, 192, 256, 384, 512}
        shares = sorted(s for s in shares if s <= 2 * CUS and s <= tiles * units)
        return [row(m, n, k, token_tiles=nt, split=s) for s in rng.sample(shares, min(per_shape, len(shares)))]
    if kind.startswith("broad"):
        block, fit = rng.choice((64, 128)) if kind == "broad blocks" else 0, []
        for nt in (4, 5, 6):
            for rows in (64, 96, 128, 160, 192, 256):
                items = _cd(m, rows) * _cd(n, 16 * nt)
                most = max(1, min(CUS // items, 16, k // 1024))
                if rows * nt <= 1024 and items * most <= 1200 and not (block and nt == 6):
                    fit += [(rows, nt, split) for split in sorted({most, max(1, most - 1), max(1, most // 2)})]
        return [row(m, n, k, block, rows=rows, token_tiles=nt, split=split) for rows, nt, split in rng.sample(fit, min(per_shape, len(fit)))]
    if kind in ("tall", "tall blocks"):
        block, fit = rng.choice((64, 128)) if kind == "tall blocks" else 0, []
        for rt in range(2, 8 if nt == 4 else 9):
            tiles = _cd(m, 16 * rt)
            most = max(1, min(CUS // tiles, 16, k // 512))
            fit += [(16 * rt, split) for split in sorted({most, max(1, most - 1), max(1, most // 2)})]
        return [row(m, n, k, block, rows=rows, token_tiles=nt, split=split) for rows, split in rng.sample(fit, min(per_shape, len(fit)))]
    block = rng.choice((64, 128)) if kind == "narrow blocks" else 0
    fit = [v for v in VARIANTS if v[3] == 1 or v[3] < 2 * nt]
    return [row(m, n, k, block, *v, split=1) for v in rng.sample(fit, min(per_shape, len(fit)))]


def _timer():
    """A function that times a launch: microseconds, the median of three runs."""
    import torch

    from . import _lib, ops
    from .quantize import nf4_codebook

    _lib.use_diagnostic_build()
    dev = torch.device("cuda:0")
    code = nf4_codebook(dev)
    pool = torch.randint(0, 256, (1 << 30,), dtype=torch.uint8, device=dev)  # weights: as many matrices as fit, in turn
    scales = torch.rand(1 << 26, device=dev) * 0.015 + 0.005
    xs = torch.randn(1 << 27, device=dev, dtype=torch.float16)
    out = torch.empty(1 << 28, dtype=torch.float16, device=dev)

    def time(r):
        m, n, k, block = r["m"], r["n"], r["k"], r["block"]
        sets = max(1, min(40, (1 << 30) // (m * k // 2)))
        q = [pool[j * (m * k // 2):(j + 1) * (m * k // 2)].view(m // 8, k // 8, 32) for j in range(sets)]
        s = [scales[:m * (k // block if block else 1)]] * sets
        x, o, cfg = xs[:n * k].view(n, k), out[:n * m].view(n, m), config_of(r)
        iters = max(10, min(100, int(4e11 / (2.0 * m * n * k + 2e9))))
        us = []
        for _ in range(3):
            ms = (ops.time_matmul_blockwise(q, s, x, code, o, m, n, k, block, config=cfg, warmup=4, iters=iters) if block else
                  ops.time_matmul(q, s, x, code, o, m, n, k, config=cfg, warmup=4, iters=iters))
            us.append(ms * 1e3 / iters)
        return round(sorted(us)[1], 2)

    return time


def measure(path, shapes, per_shape, seed, log=print, kinds=tuple(MODELS)):
    time, rng = _timer(), random.Random(seed)
    with open(path, "w", newline="") as f:
        w = csv.DictWriter(f, FIELDS)
        w.writeheader()
        for kind in kinds:
            for i in range(shapes):
                for r in launches(kind, rng, per_shape):
                    w.writerow(dict(r, us=time(r)))
                if i % 20 == 19:
                    log(f"{kind}: {i + 1} of {shapes} shapes")
                    f.flush()


def measure_again(path, kind, log=print):
    """The launches of `kind` in the file, timed again in place (that kernel has changed)."""
    rows, time = read(path), _timer()
    mine = [r for r in rows if r["kind"] == kind]
    for i, r in enumerate(mine):
        r["us"] = time(r)
        if i % 50 == 49:
            log(f"{kind}: {i + 1} of {len(mine)} launches")
    with open(path, "w", newline="") as f:
        w = csv.DictWriter(f, FIELDS)
        w.writeheader()
        w.writerows(rows)


# ---- errors and fit ---------------------------------------------------------------------------------------------------

def read(path):
    with open(path, newline="") as f:
        return [{k: v if k == "kind" else float(v) if k == "us" else int(v) for k, v in r.items()} for r in csv.DictReader(f)]


def errors(rows, model, coefficients):
    """Mean factor between predicted and measured time, less one, and the mean of predicted over measured."""
    e = [math.log(model(r, coefficients) / r["us"]) for r in rows]
    return math.exp(sum(abs(v) for v in e) / len(e)) - 1, math.exp(sum(e) / len(e))


def fit(rows, model, start):
    from scipy.optimize import least_squares

    free = [i for i, c in enumerate(start) if c != 0.0]

    def full(p):
        c = list(start)
        for i, v in zip(free, p):
            c[i] = start[i] * math.exp(v)  # (coefficients are times: they stay positive)
        return c

    res = least_squares(lambda p: [math.log(model(r, full(p)) / r["us"]) for r in rows], [0.0] * len(free), loss="soft_l1", f_scale=0.1)
    return full(res.x)


def main(argv=None):
    ap = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    ap.add_argument("csv")
    ap.add_argument("--measure", action="store_true")
    ap.add_argument("--again", metavar="KIND", help="time the launches of one kind in the file again")
    ap.add_argument("--shapes", type=int, default=100, help="random shapes per model")
    ap.add_argument("--per-shape", type=int, default=4, help="launches per shape")
    ap.add_argument("--kinds", default=",".join(MODELS), help="which models, for --measure")
    ap.add_argument("--seed", type=int, default=1)
    a = ap.parse_args(argv)
    if a.measure:
        return measure(a.csv, a.shapes, a.per_shape, a.seed, log=lambda s: print(s, flush=True), kinds=a.kinds.split(","))
    if a.again:
        return measure_again(a.csv, a.again, log=lambda s: print(s, flush=True))
    rows = read(a.csv)
    for kind, (model, coefficients) in MODELS.items():
        mine = [r for r in rows if r["kind"] == kind]
        if not mine:
            continue
        refit = fit(mine, model, coefficients)
        for name, c in (("in use", coefficients), ("refitted", refit)):
            off, bias = errors(mine, model, c)
            print(f"{kind}: {len(mine)} launches, {name}: {100 * off:.1f} % off on average, predicted / measured {bias:.3f}   "
                  + " ".join(f"{v:.4g}" for v in c))


if __name__ == "__main__":
    main()
