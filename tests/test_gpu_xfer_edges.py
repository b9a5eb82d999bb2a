"""The staging transfers of the host-pointer entries (k_xfer.hip) around the line between the
copy kernel and the copy engines (1 MB) and at sizes that are no multiple of 16 bytes: x and y
of a matmul call must arrive whole, so every row equals the row alone, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,I,O", [(1, 32, 1), (3, 32, 5), (5, 40, 777),
                                   (337, 32, 777), (338, 32, 777),           # y just below and above 1 MB
                                   (256, 32, 1024), (257, 32, 1024),         # y of exactly 1 MB, and a row more
                                   (257, 1024, 3), (256, 1024, 3)])          # x the same
def test_matmul_rows(be, S, I, O):
    rng = np.random.default_rng(S * 7 + O)
    q = rng.integers(-127, 128, (O, I)).astype(np.int8)
    sc = rng.uniform(1e-3, 2e-3, O).astype(np.float32)
    x = rng.standard_normal((S, I)).astype(np.float32)
    dq, ds = be.upload(q), be.upload(sc)
    got = be.matmul_q8(x, dq, ds, O)
    for s in sorted({0, S // 2, max(S - 2, 0), S - 1}):
        one = be.matmul_q8(x[s:s + 1], dq, ds, O)
        assert np.array_equal(got[s].view(np.uint32), one[0].view(np.uint32)), s
    dq.free(); ds.free()
    want = (x.astype(np.float64) @ q.T.astype(np.float64)) * sc
    mag = (np.abs(x).astype(np.float64) @ np.abs(q).T.astype(np.float64)) * sc
    # I roundings of 2^-24 on the products and sums, two more for the scale
    assert np.all(np.abs(got - want) <= (I + 2) * 2.0 ** -24 * mag)
