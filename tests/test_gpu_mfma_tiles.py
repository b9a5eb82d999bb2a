"""The MFMA GEMMs (k_mfma.hip) at the edges of their tiles, through lag_hip_moe_group: groups
of every size around a column (16 tokens) and a tile (16, 32 or 64 tokens by the average group
and the launch's blocks),
inputs of 1, 2, 3 and 4 quads of groups and beyond a run, outputs that end in half a row
block, every scale layout.  dot8 forms the same sums in the same order, so the bits must be
equal; dot8 itself is checked against the oracle in test_gpu_moe.py."""
import math

import numpy as np
import pytest

from sabrewing_amd.backend import Backend

pytestmark = pytest.mark.gpu
DOT8, MFMA = 1, 2


class _Layer:
    pass


def _run(be, L, x, sizes, K, gs, E=None):
    """group g: expert g (mod E), sizes[g] rows; every row is its own token (K = 1)"""
    T = sum(sizes)
    gexp, gcnt = np.arange(len(sizes), dtype=np.int32) % (E or len(sizes)), np.array(sizes, np.int32)
    gbeg = np.concatenate([[0], np.cumsum(gcnt)[:-1]]).astype(np.int32)
    perm = np.random.default_rng(7).permutation(T).astype(np.int32)      # packed row -> token
    rowof = np.empty(T, np.int32)
    rowof[perm] = np.arange(T, dtype=np.int32)
    w = np.ones((T, 1), np.float32)
    return be.moe_group(x, L, gexp, gbeg, gcnt, perm, rowof, w, K, gs)


def _parts(n, tt):
    s = math.sqrt(2 * n)
    k = int((n - 4 * s) / tt) if n > 4 * s else 0
    e, k = 1.0 + k, k + 1
    while k * tt < n + 4 * s:
        e, k = e + 0.5 * math.erfc((k * tt + 0.5 - n) / s), k + 1
    return e


def tile_width(sizes, D, I, known=True):
    """the launch rule (sw_mf_cols): by the average group, narrower where the rounds of blocks
    on the CUs times a block's time say so; known: the host knows the groups' sizes"""
    T, G = sum(sizes), len(sizes)
    top = 16 if T <= 9 * G else 32 if T <= 22 * G else 64
    if top == 16:
        return top
    parts = lambda tt: sum(-(-n // tt) for n in sizes) if known else G * _parts(T / G, tt)
    cols, best, limit = parts(16), top, 0.0
    for tt, fill, col in ((64, 3, (62, 68, 85, 115)), (32, 2.5, (50, 64)), (16, 2, (45,))):
        if tt > top:
            continue
        tiles = parts(tt)
        c = float(np.interp(cols / tiles, range(1, tt // 16 + 1), col))
        t = sum(max(1, math.ceil(tiles * nb / 256 - (0 if known else 0.01))) * (fill + K / 4096 * c) for K, nb in ((D, I // 128), (I, -(-D // 256))))
        if tt == top:
            limit = 0.95 * t
        elif t < limit:
            best, limit = tt, t
    return best


def wide(sizes, D, I):
    """the groups repeated until their launch takes the widest tile their average allows"""
    T, G = sum(sizes), len(sizes)
    top = 16 if T <= 9 * G else 32 if T <= 22 * G else 64
    return next(sizes * r for r in range(1, 400) if tile_width(sizes * r, D, I) == top)


@pytest.mark.parametrize("gs", [0, 32, 64, 128])
@pytest.mark.parametrize("D,I", [(128, 128), (256, 384), (384, 256), (640, 128), (1152, 512)])
@pytest.mark.parametrize("sizes,tt", [([1, 16, 2, 15, 3], 16), ([17, 16, 31, 1, 32], 32), ([33, 64, 63, 16, 5], 64),
                                      ([65, 129, 48, 1, 80], 64)], ids=["cols16", "cols32", "cols64", "split"])
@pytest.mark.parametrize("many", [False, True], ids=["few", "many"])
def test_mfma_tiles_equal_dot8(be: Backend, gs, D, I, sizes, tt, many):
    rng = np.random.default_rng(D + I + gs)
    E, n = len(sizes), lambda K: K // gs if gs else 1
    if many:
        sizes = wide(sizes, D, I)
    assert tile_width(sizes, D, I) == (tt if many else 16)
    L = _Layer()
    L.D, L.I = D, I
    q = lambda r, K: be.upload(rng.integers(0, 256, (r, K // 2), dtype=np.uint8))
    s = lambda r, K: be.upload(rng.uniform(1e-3, 4e-3, (r, n(K))).astype(np.float32))
    L.gu_q, L.gu_s, L.dn_q, L.dn_s = q(E * 2 * I, D), s(E * 2 * I, D), q(E * D, I), s(E * D, I)
    x = rng.standard_normal((sum(sizes), D)).astype(np.float32) * rng.choice([1e-3, 1.0, 30.0], (sum(sizes), 1)).astype(np.float32)
    x[:, :32] = 0.0                                   # a zero group, and a token of zeros
    x[1] = 0.0
    out = {}
    for mode in (DOT8, MFMA):
        prev = be.set_grouped_kernel(mode)
        try:
            out[mode] = _run(be, L, x, sizes, 1, gs, E)
        finally:
            be.set_grouped_kernel(prev)
    for b in (L.gu_q, L.gu_s, L.dn_q, L.dn_s):
        b.free()
    assert np.isfinite(out[DOT8]).all()
    assert np.array_equal(out[MFMA].view(np.uint32), out[DOT8].view(np.uint32))


def _row_blocks(D, I, sizes):
    """the down's row blocks per block: up to four while that leaves 1024 blocks"""
    tt, nrb = tile_width(sizes, D, I), -(-D // 256)
    tiles = sum(-(-n // tt) for n in sizes)
    return next((r for r in (4, 2) if nrb % r == 0 and tiles * (nrb // r) >= 1024), 1)


# (D, groups, rows per group, tile width, row blocks per block): D of 3.5 and 7.5 row blocks
MANY = [(1920, 540, (1, 9), 16, 4), (1920, 280, (1, 9), 16, 2), (1920, 560, (8, 23), 32, 4), (1920, 360, (8, 23), 32, 2),
        (1920, 560, (20, 40), 64, 4), (1920, 256, (24, 48), 64, 2), (896, 640, (8, 23), 32, 2), (896, 540, (1, 9), 16, 2)]


@pytest.mark.parametrize("gs", [0, 32])
@pytest.mark.parametrize("I", [128, 384, 512])
@pytest.mark.parametrize("D,G,lohi,tt,r", MANY, ids=lambda v: str(v).replace(" ", ""))
def test_down_over_several_row_blocks(be: Backend, D, G, lohi, tt, r, I, gs):
    """many groups: a down block runs 2 or 4 row blocks through one pipeline (the digits of a
    chunk again for each, the next row block's weights ahead), with 1, 3 and 4 quads of inputs
    (a half-filled last chunk where a chunk holds two) and outputs that end in half a row block"""
    rng = np.random.default_rng(D + I + G)
    sizes = [int(n) for n in rng.integers(*lohi, G)]
    assert (tile_width(sizes, D, I), _row_blocks(D, I, sizes)) == (tt, r)
    E, n = 4, lambda K: K // gs if gs else 1
    L = _Layer()
    L.D, L.I = D, I
    q = lambda rows, K: be.upload(rng.integers(0, 256, (rows, K // 2), dtype=np.uint8))
    s = lambda rows, K: be.upload(rng.uniform(1e-3, 4e-3, (rows, n(K))).astype(np.float32))
    L.gu_q, L.gu_s, L.dn_q, L.dn_s = q(E * 2 * I, D), s(E * 2 * I, D), q(E * D, I), s(E * D, I)
    x = rng.standard_normal((sum(sizes), D), dtype=np.float32)
    out = {}
    for mode in (DOT8, MFMA):
        prev = be.set_grouped_kernel(mode)
        try:
            out[mode] = _run(be, L, x, sizes, 1, gs, E)
        finally:
            be.set_grouped_kernel(prev)
    for b in (L.gu_q, L.gu_s, L.dn_q, L.dn_s):
        b.free()
    assert np.isfinite(out[DOT8]).all() and (out[DOT8] != 0).any()
    assert np.array_equal(out[MFMA].view(np.uint32), out[DOT8].view(np.uint32))
