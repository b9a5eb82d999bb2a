"""The host-activation matmuls where their two kernels meet (k_lanes.hip): rows in whole
16-byte pieces are streamed by waves, everything else takes the general tiles.  Inputs around
a step (128, 256 or 512 columns by the weight type), an x chunk (512 columns) and the scalar
tail, outputs around a wave's 4 rows and a block's 16; a weight address off by one element
takes the general kernel, and so do short rows of many outputs.  With few outputs the streamed
kernel runs a token at a time, whatever the batch; test_widths has enough of them for its
passes of 1, 2, 4 and 8.  All bit for bit the oracle's, whose matmuls are pinned to the
compiled reference."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SHAPES = [(32, 1), (64, 5), (96, 16), (160, 17), (512, 3), (528, 20), (544, 33), (1024, 18), (1056, 7), (1504, 67)]
TOKENS = [1, 2, 3, 4, 7, 8, 9, 17]


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


class _At:
    def __init__(self, buf, off):
        self.p = int(buf) + off

    def __int__(self):
        return self.p


def _x(rng, S, I):
    x = rng.standard_normal((S, I)).astype(np.float32)
    x[0, ::7] = 0.0
    x[-1, 1::5] *= np.float32(1e-30)                  # products below the normal range
    return x


@pytest.mark.parametrize("I,O", SHAPES + [(40, 9), (536, 19)])
def test_bf16(be, orc, I, O):
    rng = np.random.default_rng(I * 131 + O)
    Wb = orc.to_bf16(rng.standard_normal((O, I)).astype(np.float32) * np.float32(0.02)).reshape(O, I)
    Wb[0, :3] = [1, 0x8001, 0x7F]                     # denormal weights
    pad = np.zeros(O * I + 1, np.uint16)
    pad[1:] = Wb.reshape(-1)
    d0, d1 = be.upload(Wb), be.upload(pad)
    for S in TOKENS:
        x = _x(rng, S, I)
        for got in (be.matmul_bf16(x, d0, O), be.matmul_bf16(x, _At(d1, 2), O)):
            assert np.array_equal(bits(got), bits(orc.matmul_bf16(x, Wb))), (S, I, O)
        for got in (be.matmul_bf16_rx(x, d0, O), be.matmul_bf16_rx(x, _At(d1, 2), O)):
            assert np.array_equal(bits(got), bits(orc.matmul_bf16_rx(x, Wb))), (S, I, O)
    d0.free(); d1.free()


@pytest.mark.parametrize("I,O", SHAPES + [(1040, 6)])
def test_q8(be, orc, I, O):
    rng = np.random.default_rng(I * 137 + O)
    q = rng.integers(-127, 128, (O, I)).astype(np.int8)
    sc = rng.uniform(1e-3, 2e-3, O).astype(np.float32)
    pad = np.zeros(O * I + 1, np.int8)
    pad[1:] = q.reshape(-1)
    d0, d1, ds = be.upload(q), be.upload(pad), be.upload(sc)
    for S in TOKENS:
        x = _x(rng, S, I)
        for got in (be.matmul_q8(x, d0, ds, O), be.matmul_q8(x, _At(d1, 1), ds, O)):
            assert np.array_equal(bits(got), bits(orc.matmul_q8(x, q, sc, 0))), (S, I, O)
    for b in (d0, d1, ds):
        b.free()


@pytest.mark.parametrize("I,O", SHAPES)
def test_q4(be, orc, I, O):
    rng = np.random.default_rng(I * 139 + O)
    p = rng.integers(0, 256, (O, I // 2), dtype=np.uint8)
    sc = rng.uniform(1e-3, 2e-3, O).astype(np.float32)
    pad = np.zeros(O * I // 2 + 1, np.uint8)
    pad[1:] = p.reshape(-1)
    d0, d1, ds = be.upload(p), be.upload(pad), be.upload(sc)
    for S in TOKENS:
        x = _x(rng, S, I)
        for got in (be.matmul_q4(x, d0, ds, O, 0), be.matmul_q4(x, _At(d1, 1), ds, O, 0)):
            assert np.array_equal(bits(got), bits(orc.matmul_q4(x, p, sc))), (S, I, O)
    for b in (d0, d1, ds):
        b.free()


def _width(O, S):
    """tokens per pass of the streamed kernel: the most that leave 512 blocks"""
    ts = 8 if S >= 8 else 4 if S >= 3 else S
    while ts > 1 and -(-O // 16) * -(-S // ts) < 512:
        ts //= 2
    return ts


def _short(O, S, I):
    """rows too short, for that many blocks, to be streamed"""
    ts = 16 if S >= 16 else 8 if S >= 8 else 4 if S >= 4 else 1
    nb = -(-O // 16) * -(-S // ts)
    return nb >= 512 and I <= min(nb // 6, 224 + nb // 40)


WIDE_O = 8195                                         # 513 blocks a pass: every width is reached
WIDE_S = [1, 2, 3, 4, 7, 8, 9, 17]                    # full passes, and passes with tokens past the batch


@pytest.mark.parametrize("kind,I", [("bf16", 288), ("bf16", 536), ("bf16", 1056),
                                    ("bf16_rx", 288), ("bf16_rx", 544), ("bf16_rx", 1056),
                                    ("q8", 272), ("q8", 528), ("q8", 1040),
                                    ("q4", 288), ("q4", 544), ("q4", 1056)])
def test_widths(be, orc, kind, I):
    """each width of the streamed kernel on full and partial steps and chunks"""
    assert [_width(WIDE_O, S) for S in WIDE_S] == [1, 2, 4, 4, 4, 8, 8, 8]
    assert not any(_short(WIDE_O, S, I) for S in WIDE_S)
    _against_oracle(be, orc, kind, I)


@pytest.mark.parametrize("kind,I", [("bf16", 32), ("bf16", 160), ("bf16_rx", 32), ("bf16_rx", 160),
                                    ("q8", 32), ("q8", 160), ("q4", 32), ("q4", 160)])
def test_short_rows(be, orc, kind, I):
    """rows of whole pieces on both sides of the line to the general kernel"""
    assert {_short(WIDE_O, S, I) for S in WIDE_S} == ({True} if I == 32 else {True, False})
    _against_oracle(be, orc, kind, I)


def _against_oracle(be, orc, kind, I):
    O = WIDE_O
    rng = np.random.default_rng(I * 149 + len(kind))
    sc = rng.uniform(1e-3, 2e-3, O).astype(np.float32)
    if kind == "q8":
        W = rng.integers(-127, 128, (O, I)).astype(np.int8)
    elif kind == "q4":
        W = rng.integers(0, 256, (O, I // 2), dtype=np.uint8)
    else:
        W = orc.to_bf16(rng.standard_normal((O, I)).astype(np.float32) * np.float32(0.02)).reshape(O, I)
        W[0, :3] = [1, 0x8001, 0x7F]
    d, ds = be.upload(W), be.upload(sc)
    run, ref = {"bf16": (lambda x: be.matmul_bf16(x, d, O), lambda x: orc.matmul_bf16(x, W)),
                "bf16_rx": (lambda x: be.matmul_bf16_rx(x, d, O), lambda x: orc.matmul_bf16_rx(x, W)),
                "q8": (lambda x: be.matmul_q8(x, d, ds, O), lambda x: orc.matmul_q8(x, W, sc, 0)),
                "q4": (lambda x: be.matmul_q4(x, d, ds, O, 0), lambda x: orc.matmul_q4(x, W, sc))}[kind]
    for S in WIDE_S:
        x = _x(rng, S, I)
        assert np.array_equal(bits(run(x)), bits(ref(x))), S
    d.free(); ds.free()


@pytest.mark.parametrize("S", [8 * 65535, 8 * 65535 + 1])
def test_most_tokens(be, orc, S):
    """the last row count whose passes of 8 tokens would fit a grid's second dimension (65535),
    and one more (such short rows take the general kernel's passes of 16 either way)"""
    I = 32
    rng = np.random.default_rng(S)
    q = rng.integers(-127, 128, (1, I)).astype(np.int8)
    sc = rng.uniform(1e-3, 2e-3, 1).astype(np.float32)
    x = rng.standard_normal((S, I), dtype=np.float32)
    dq, ds = be.upload(q), be.upload(sc)
    got = be.matmul_q8(x, dq, ds, 1)
    dq.free(); ds.free()
    assert np.array_equal(bits(got), bits(orc.matmul_q8(x, q, sc, 0)))
