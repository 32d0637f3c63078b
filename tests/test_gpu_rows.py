"""Activation producer rows (smq_row_quantize, smq_norm_quantize, smq_quantize_q8_rows) against the oracle's row_work,
bit for bit, at the edges of their kernels: whole-block rows (one flat run) and ragged ones, unaligned buffers, the
stored f32 row in place, and RMSNorm sums of every chain length."""
import numpy as np
import pytest

from checks import assert_same_f32, say
from smq_pkg import smq, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    assert smq.init(0) == "gfx950"
    smq.kernels_set_fast(False)
    yield


def dev(a):
    return smq.DeviceBuffer.from_array(a)


@pytest.mark.parametrize("rows,n,shift", [(1, 32, 0), (3, 896, 0), (33, 4864, 0), (5, 96, 0), (3, 896, 4), (7, 100, 0),
                                          (2, 12288, 0), (129, 64, 0)])
@pytest.mark.parametrize("act", [0, 1, 2])
def test_rows(orc, rows, n, shift, act):
    say("rows", rows, n, shift, act)
    nb = (n + 31) // 32
    x, g = synth.normal(71, rows * n, 3.0), synth.normal(72, rows * n, 4.0)
    g[:5] = (0.0, -0.0, 88.5, -104.5, 1e-30)
    xb, gb = smq.DeviceBuffer(x.nbytes + 16), smq.DeviceBuffer(g.nbytes + 16)
    xb.upload(x, shift)
    gb.upload(g, shift)
    d, q = smq.DeviceBuffer(rows * nb * 4), smq.DeviceBuffer(rows * nb * 32)
    gate = gb.at(shift) if act else None
    ok, wy, wd, wq = orc.row_work(x, rows, n, gate=g if act else None, gelu=act == 2)
    assert ok
    for y in (None, xb.at(shift)):  # the second pass stores the f32 row over its source
        smq.row_quantize(xb.at(shift), rows, n, d, q, gate=gate, act=act, y=y)
        smq.numeric_check()
        assert_same_f32(d.download(np.float32), wd, "scales")
        assert np.array_equal(q.download(np.int8), wq)
    assert_same_f32(xb.download(np.float32, rows * n, shift), wy, "f32 row")
    if act == 0:
        smq.quantize_q8_rows(gb.at(shift), rows, n, d, q)
        _, wd, wq = orc.quantize_q8(g.reshape(rows, n))
        assert_same_f32(d.download(np.float32), wd.reshape(-1), "scales of quantize_q8_rows")
        assert np.array_equal(q.download(np.int8), wq.reshape(-1))


@pytest.mark.parametrize("shift", [1, 2, 4])
@pytest.mark.parametrize("act", [0, 1, 2])
def test_rows_unaligned_output(orc, shift, act):
    """Whole-block rows whose int8 output starts at any byte."""
    say("rows, unaligned output", shift, act)
    rows, n = 3, 896
    x, g = synth.normal(75, rows * n, 3.0), synth.normal(76, rows * n, 4.0)
    d, q = smq.DeviceBuffer(rows * n // 32 * 4), smq.DeviceBuffer(rows * n + 8)
    q.fill(0x5A)
    xb, gb = dev(x), dev(g)
    smq.row_quantize(xb, rows, n, d, q.at(shift), gate=gb if act else None, act=act)
    smq.numeric_check()
    ok, _, wd, wq = orc.row_work(x, rows, n, gate=g if act else None, gelu=act == 2)
    assert ok
    assert_same_f32(d.download(np.float32), wd, "scales")
    got = q.download(np.int8)
    assert np.array_equal(got[shift:shift + rows * n], wq.reshape(-1))
    assert (got[:shift] == 0x5A).all() and (got[shift + rows * n:] == 0x5A).all()


@pytest.mark.parametrize("n", [255, 257, 640, 1024, 1025, 1536, 1537, 2048, 2049, 3000, 4096, 4100, 8192, 16384])
def test_norm_chains(orc, n):
    say("norm chain", n)
    x, w = synth.normal(73, 2 * n, 2.0), 1.0 + synth.normal(74, n, 0.1)
    xb, wb = dev(x), dev(w.astype(np.float32))
    nb = (n + 31) // 32
    d, q = smq.DeviceBuffer(2 * nb * 4), smq.DeviceBuffer(2 * nb * 32)
    smq.norm_quantize(xb, wb, 1e-6, 2, n, None, d, q)
    smq.numeric_check()
    ok, _, wd, wq = orc.row_work(x, 2, n, norm=w.astype(np.float32), eps=1e-6)
    assert ok
    assert_same_f32(d.download(np.float32), wd, "scales")
    assert np.array_equal(q.download(np.int8), wq)
