"""The unscaled shared expert of a batch on its own (k_shared.hip): every kernel its launch
rule picks (split-K with one and two row tiles, the LDS tiles) and both sides of each line,
against the single-token path (the decode stages' jobs), bit for bit: all form the same
chains and fold the same segments in the same order."""
import numpy as np
import pytest

from oracle import synth
from sabrewing_amd import configs as cf
from sabrewing_amd.backend import DeviceLayer, desc_of

pytestmark = pytest.mark.gpu
MFMA = 2          # the experts on the MFMA: the shared expert runs in launches of its own

# (D, Is): segments of 1 group; 4 segments of 3 groups; 4 segments of 9 in the down; a down of
# 65 to 128 tokens in tiles, and one whose K split runs in two rounds on the CUs
SHAPES = [(256, 1024), (384, 1024), (256, 1152), (1536, 512), (1536, 1024)]


@pytest.mark.parametrize("D,Is", SHAPES)
@pytest.mark.parametrize("S_", [17, 64, 65, 128, 129, 181, 256, 257, 321])
def test_shared_batch_equals_single_token(be, orc, D, Is, S_):
    cfg = cf.scaled(cf.C2, D=D, E=8, K=2, I=128, Is=Is)
    L = synth.make_layer(orc, cfg, 91)
    x = synth.make_x(orc, cfg, 92, S_)
    base = synth.make_x(orc, cfg, 93, S_)
    dl = DeviceLayer.from_host(be, cfg, L)
    prev = be.set_grouped_kernel(MFMA)
    try:
        got = be.moe_block(desc_of(cfg), dl.weights(), x, base)
        rows = sorted({0, 15, 16, S_ // 2, S_ - 2, S_ - 1})
        one = np.stack([be.moe_block(desc_of(cfg), dl.weights(), x[s:s + 1], base[s:s + 1])[0] for s in rows])
    finally:
        be.set_grouped_kernel(prev)
    dl.free()
    assert np.array_equal(got[rows].view(np.uint32), one.view(np.uint32))
