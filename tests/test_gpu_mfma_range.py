"""The MFMA GEMMs (k_mfma.hip) give dot8's bits over the whole range of scales and inputs, also
where dot8's term acc (s xf) and an equal term in another order, (acc s) xf, round differently:
products of scale and factor below the normal range, zero, negative and denormal scales, acc s
beyond the largest float, terms that overflow, NaN (any NaN for a NaN) -- for every scale
layout and tile width, when one token and one expert out of many hold such values and when
all do."""
import numpy as np
import pytest

from sabrewing_amd.backend import Backend
from test_gpu_mfma_tiles import tile_width, wide

pytestmark = pytest.mark.gpu
DOT8, MFMA = 1, 2
E = 5
D, I = 1152, 384                    # 9 and 3 quads of input groups: a short last run each


def _spread(rng, shape, lo, hi):
    return np.exp2(rng.uniform(lo, hi, shape)).astype(np.float32)


# what is out of the ordinary: (x, gate/up scales, down scales) of a case, per whole group of
# 32 inputs (x) and per scale; the ordinary values are x ~ N(0, 1), scales in [1e-3, 4e-3]
def _tiny_x(rng, x, gs_, ds_):      # group maxima from 2^-149 to 2^-60: s xf denormal, or xf itself
    x *= np.repeat(_spread(rng, (x.shape[0], D // 32), -150, -60), 32, axis=1)


def _edge_x(rng, x, gs_, ds_):      # s xf within a few powers of two of the smallest normal number
    x *= np.repeat(_spread(rng, (x.shape[0], D // 32), -100, -88), 32, axis=1)
    gs_ *= np.float32(2.0 ** 0.5)


def _tiny_h(rng, x, gs_, ds_):      # the down's inputs: h ~ x^2
    x *= np.repeat(_spread(rng, (x.shape[0], 1), -62, -40), D, axis=1)


def _tiny_s(rng, x, gs_, ds_):      # gate scales denormal, some zero, some negative, beside large up scales
    g = gs_.reshape(-1, 2, I, gs_.shape[1])
    g[:, 0] *= _spread(rng, g[:, 0].shape, -146, -110)
    g[:, 0][rng.random(g[:, 0].shape) < 0.2] = 0.0
    g[:, 0][rng.random(g[:, 0].shape) < 0.2] *= -1.0
    g[:, 1] *= np.float32(2.0 ** 100)


def _tiny_ds(rng, x, gs_, ds_):     # the same in the down
    ds_ *= _spread(rng, ds_.shape, -146, -100)
    ds_[rng.random(ds_.shape) < 0.2] = 0.0
    ds_[rng.random(ds_.shape) < 0.2] *= -1.0


def _zero_s(rng, x, gs_, ds_):
    gs_[3::7] = 0.0
    ds_[5::11] = 0.0


def _huge_s(rng, x, gs_, ds_):      # acc s overflows, acc (s xf) does not
    x *= np.float32(2.0 ** -100)
    gs_ *= np.float32(2.0 ** 110)


def _huge_x(rng, x, gs_, ds_):      # terms up to and beyond the largest float
    x *= np.repeat(_spread(rng, (x.shape[0], D // 32), 90, 125), 32, axis=1)
    gs_ *= _spread(rng, gs_.shape, 0, 8)


def _nan(rng, x, gs_, ds_):
    x[::3, 40] = np.nan
    x[1::3, 100] = np.inf


KINDS = {f.__name__[1:]: f for f in (_tiny_x, _edge_x, _tiny_h, _tiny_s, _tiny_ds, _zero_s, _huge_s, _huge_x, _nan)}


def _run(be, b, x, sizes, gs):
    T = sum(sizes)

    class L:
        gu_q, gu_s, dn_q, dn_s = b
    L.D, L.I = D, I
    gcnt = np.array(sizes, np.int32)
    gbeg = np.concatenate([[0], np.cumsum(gcnt)[:-1]]).astype(np.int32)
    perm = np.random.default_rng(7).permutation(T).astype(np.int32)
    rowof = np.empty(T, np.int32)
    rowof[perm] = np.arange(T, dtype=np.int32)
    gexp = np.arange(len(sizes), dtype=np.int32) % E
    return be.moe_group(x, L, gexp, gbeg, gcnt, perm, rowof, np.ones((T, 1), np.float32), 1, gs)


def _equal(a, b):
    na, nb = np.isnan(a), np.isnan(b)
    return np.array_equal(na, nb) and np.array_equal(a.view(np.uint32)[~na], b.view(np.uint32)[~nb])


@pytest.mark.parametrize("gs", [0, 32, 64, 128])
@pytest.mark.parametrize("sizes,tt", [([1, 16, 2, 15, 3], 16), ([17, 16, 31, 1, 32], 32), ([33, 64, 63, 81, 5], 64)],
                         ids=["cols16", "cols32", "cols64"])
@pytest.mark.parametrize("kind", list(KINDS))
def test_bits_outside_the_ordinary(be: Backend, kind, sizes, tt, gs):
    sizes = wide(sizes, D, I)
    assert tile_width(sizes, D, I) == tt
    T = sum(sizes)
    rng = np.random.default_rng(gs + T)
    n = lambda K: K // gs if gs else 1
    q = lambda r, K: rng.integers(0, 256, (r, K // 2), dtype=np.uint8)
    s = lambda r, K: rng.uniform(1e-3, 4e-3, (r, n(K))).astype(np.float32)
    gq, gsc, dq, dsc, x0 = q(E * 2 * I, D), s(E * 2 * I, D), q(E * D, I), s(E * D, I), \
        rng.standard_normal((T, D)).astype(np.float32)
    seen = False
    for whole in (False, True):     # a few tokens and one expert, then every one
        x, a, b = x0.copy(), gsc.copy(), dsc.copy()
        if whole:
            with np.errstate(over="ignore"):
                KINDS[kind](rng, x, a, b)
        else:
            tok = np.arange(0, T, 5)
            xs, as_, bs = x[tok], a[2 * 2 * I:3 * 2 * I], b[2 * D:3 * D]
            with np.errstate(over="ignore"):
                KINDS[kind](rng, xs, as_, bs)
            x[tok] = xs             # (as_ and bs are views)
        bufs = [be.upload(v) for v in (gq, a, dq, b)]
        out = {}
        for mode in (DOT8, MFMA):
            prev = be.set_grouped_kernel(mode)
            try:
                out[mode] = _run(be, bufs, x, sizes, gs)
            finally:
                be.set_grouped_kernel(prev)
        for v in bufs:
            v.free()
        seen |= bool((np.isfinite(out[DOT8]) & (out[DOT8] != 0)).any())
        assert _equal(out[MFMA], out[DOT8]), ("all" if whole else "some", int((out[MFMA] != out[DOT8]).sum()))
    assert seen
