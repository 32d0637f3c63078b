"""2-16 tokens (k_gemv_few and the tiles beside its rule) against the CPU oracle, bit for bit: both formats and
orders, ragged rows, one and several chunks of a row, every count of passes, item edges, bias, residual add and
non-finite values."""
import numpy as np
import pytest

from checks import q5_random
from patterns import LcgUniform
from smq_pkg import smq, synth
from test_gpu_parity import Q5B, Q8B, assert_same_f32, bits, gpu_quantize, run_gemm, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    assert smq.init(0) == "gfx950"
    smq.kernels_set_fast(False)
    smq.kernels_select()
    yield


SHAPES = [  # rows, blocks (Q5 rows of an odd count take the generic kernel), tokens
    (1, 12, 2),       # the shortest row of one pass, one row
    (13, 28, 4), (77, 28, 5),   # eight rows per workgroup, idle tasks, a second pass of one token
    (43, 32, 3), (101, 34, 8),  # Q8's one whole chunk, then two chunks with four rows
    (67, 64, 16), (29, 66, 13), # Q5's one whole chunk (four passes), then two chunks
    (509, 152, 9),    # three passes, a partial last Q8 chunk
    (45, 280, 12), (2053, 130, 7),  # several chunks; Q5 past 2048 rows: eight rows with three chunks
    (4101, 28, 6), (8201, 48, 2), (8201, 48, 6), (8201, 48, 11),  # beside the rule: tiles of 8 tokens, of 16 over four waves
    (16403, 30, 7), (16403, 30, 15),   # more 32-row tiles than two per CU
]


@pytest.mark.parametrize("fast", [False, True])
@pytest.mark.parametrize("q5", [False, True])
@pytest.mark.parametrize("rows,nb,ntok", SHAPES)
def test_few_tokens(orc, rows, nb, ntok, q5, fast):
    say("few tokens", rows, nb, ntok, q5, fast)
    cols, stride = nb * 32, rows + 3
    w = (q5_random(71, rows, cols) if q5 else synth.q8_weights(71, rows, cols)).reshape(-1)
    x = synth.activations(72, ntok, cols)
    got, xd, xq = run_gemm(w, nb * (Q5B if q5 else Q8B), x, rows, ntok, nb, q5, stride, fast)
    want = orc.gemm(w, nb * (Q5B if q5 else Q8B), xd, xq, rows, ntok, nb, stride=stride, q5=q5, fast=fast)
    m = np.zeros(ntok * stride, bool)
    m.reshape(ntok, stride)[:, :rows] = True
    assert_same_f32(got[m], want[m], "few")
    assert np.all(bits(got[~m]) == 0xFFFFFFFF), "wrote outside the output rows"


@pytest.mark.parametrize("q5", [False, True])
@pytest.mark.parametrize("ntok", [3, 7, 14])
def test_few_tokens_items(orc, q5, ntok):
    g = LcgUniform(47)
    cols = 2112
    nb, bb = cols // 32, Q5B if q5 else Q8B
    say("few tokens items", q5, ntok)
    dbuf, qbuf, xd, xq = gpu_quantize(synth.activations(48, ntok, cols))
    items, wants = [], []
    for i, rows in enumerate([33, 100, 7, 64]):
        w = (q5_random(80 + i, rows, cols) if q5 else synth.q8_weights(80 + i, rows, cols)).reshape(-1)
        bias = g.uniform(-0.1, 0.1, rows) if i % 2 == 0 else None
        acc = i % 3 == 1
        y0 = g.uniform(-1, 1, ntok * rows).astype(np.float32) if acc else np.zeros(ntok * rows, np.float32)
        ok, y = orc.mat_item(w, nb * bb, rows, bias, xd, xq, ntok, nb, q5=q5)
        assert ok
        wants.append(y0 + y if acc else y)
        items.append((smq.QMat(smq.DeviceBuffer.from_array(w), rows, cols, smq.DTYPE_Q5 if q5 else smq.DTYPE_Q8),
                      smq.DeviceBuffer.from_array(bias) if bias is not None else None,
                      smq.DeviceBuffer.from_array(y0), acc))
    smq.matmul(items, dbuf, qbuf, ntok)
    smq.numeric_check()
    for i, (it, want) in enumerate(zip(items, wants)):
        assert_same_f32(it[2].download(np.float32), want, f"item {i}")
    if not q5:
        w = synth.q8_weights(7, 40, cols).reshape(-1)
        w[36 * nb * 3:36 * nb * 3 + 4] = np.array([np.inf], np.float32).view(np.uint8)  # row 3, block 0
        yb = smq.DeviceBuffer(ntok * 40 * 4)
        smq.matmul([(smq.QMat(smq.DeviceBuffer.from_array(w), 40, cols), None, yb)], dbuf, qbuf, ntok)
        with pytest.raises(smq.SmqError) as e:
            smq.numeric_check()
        assert e.value.status == smq.SM_ERR_NUMERIC
