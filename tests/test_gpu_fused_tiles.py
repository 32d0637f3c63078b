"""The fused decode GEMV over many tiles per workgroup (rows of one chunk: the activation in registers, two tiles in
flight, the gated products in groups of 64 tiles) and over several chunks, against the CPU oracle, bit for bit."""
import numpy as np
import pytest

from smq_pkg import smq, synth
from test_gpu_fused import Q5, Q8, assert_same_f32, dev, expect_items, say, weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    assert smq.init(0) == "gfx950"
    smq.kernels_set_fast(False)
    smq.kernels_select()
    yield


def norm_act(orc, cols):
    nb = (cols + 31) // 32
    x, w = synth.normal(41 + cols, cols), synth.normal(42 + cols, cols, 0.2) + 1.0
    ok, _, d, q = orc.row_work(x, 1, cols, norm=w, eps=1e-6)
    assert ok
    return smq.act(smq.ACT_NORM, cols, x=dev(x), norm=dev(w), eps=1e-6, xd_scratch=smq.DeviceBuffer(nb * 4),
                   xq_scratch=smq.DeviceBuffer(nb * 32)), d, q


@pytest.mark.parametrize("cols,rows,dtype,glu", [
    (64, 300003, Q5, 1),    # more than 64 tiles of four rows per workgroup, a partial last tile
    (96, 300001, Q8, 2),
    (1536, 8960, Q5, 1), (1504, 1, Q8, 1), (1024, 4099, Q5, 2),
    (2048, 2050, Q8, 1),    # two rows of each matrix per tile
    (3200, 1031, Q8, 1), (4864, 1030, Q5, 1),   # one row of each
    (4864, 515, Q8, 1),     # several chunks
])
def test_fused_glu_tiles(orc, cols, rows, dtype, glu):
    say("fused glu tiles", cols, rows, dtype, glu)
    act, d, q = norm_act(orc, cols)
    wg, wu = weights(43, rows, cols, dtype), weights(44, rows, cols, dtype)
    h = smq.DeviceBuffer(rows * 4)
    smq.matmul_glu(smq.QMat(dev(wg), rows, cols, dtype), smq.QMat(dev(wu), rows, cols, dtype), act, glu, h,
                   gate_scratch=smq.DeviceBuffer(rows * 4))
    smq.numeric_check()
    g, u = expect_items(orc, [(wg, rows, dtype, None, None), (wu, rows, dtype, None, None)], d, q, cols)
    ok, want, _, _ = orc.row_work(u, 1, rows, gate=g, gelu=glu == 2)
    assert ok
    assert_same_f32(h.download(np.float32), want, "h")


@pytest.mark.parametrize("cols,rows,dtype", [
    (1536, (8203, 33, 1001), Q5), (576, (20001, 7), Q8), (2048, (4099, 1), Q8), (4864, (2051, 5), Q5), (8192, (300,), Q8),
])
def test_fused_store_tiles(orc, cols, rows, dtype):
    say("fused store tiles", cols, rows, dtype)
    act, d, q = norm_act(orc, cols)
    items, spec = [], []
    for i, r in enumerate(rows):
        w, bias, prior = weights(45 + i, r, cols, dtype), synth.normal(46 + i, r), synth.normal(49 + i, r)
        items.append((smq.QMat(dev(w), r, cols, dtype), dev(bias), dev(prior), True))
        spec.append((w, r, dtype, bias, prior))
    smq.matmul_act(items, act)
    smq.numeric_check()
    for it, want in zip(items, expect_items(orc, spec, d, q, cols)):
        assert_same_f32(it[2].download(np.float32), want, "y")
