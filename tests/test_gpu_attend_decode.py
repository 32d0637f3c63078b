"""One token's attention in two launches (scores, then values) at head sizes other than 64, and the value sums past
640 positions, against the oracle's attend_f32, bit for bit: eager, in a captured graph (which owns its score
workspace), and on another stream (one launch, no workspace)."""
import numpy as np
import pytest
import torch

from checks import assert_same_f32, say
from smq_pkg import smq, synth
from test_gpu_decoder import attend_expect, dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    assert smq.init(0) == "gfx950"
    smq.kernels_set_fast(False)
    smq.kernels_select()
    yield


CASES = [  # heads, kv_heads, hd, window, context, positions
    (4, 2, 32, 0, 300, (0, 31, 246, 247, 255, 256, 299)), # the smallest head: both sides of the rule (graphs: from 0), tiles of 32 scores
    (6, 2, 96, 0, 700, (63, 638, 639, 640, 641, 699)), # one chunk of values against the long form
    (12, 2, 128, 0, 1400, (767, 768, 769, 1023, 1024, 1279, 1280)), # both buffers, chunk edges
    (16, 1, 256, 0, 300, (255, 256, 299)),             # the largest head, 16 of them per group
    (17, 1, 32, 0, 64, (63,)),                         # 17 per group: the one launch
    (4, 4, 160, 700, 2000, (698, 699, 700, 1999)),     # a window that starts in the middle of a tile
    (2, 1, 128, 0, 16384, (16383,)),                   # the longest context
    (14, 2, 64, 0, 1400, (639, 640, 767, 768, 1024, 1399)), # head_dim 64 past one chunk
    (2, 1, 64, 650, 16384, (648, 649, 650, 16383)),
]


@pytest.mark.parametrize("heads,kv_heads,hd,window,context,positions", CASES)
def test_attend_decode(orc, heads, kv_heads, hd, window, context, positions):
    say("attend decode", heads, kv_heads, hd, window, context, positions)
    qd, kd = heads * hd, kv_heads * hd
    nb = qd // 32
    q = synth.normal(51, qd, 2.0).reshape(1, qd)
    keys = synth.normal(52, context * kd).reshape(context, kd)
    values = synth.normal(53, context * kd).reshape(context, kd)
    qb, kb, vb = dev(q), dev(keys), dev(values)
    shape = smq.attn_shape(heads, kv_heads, hd, hd // 2, window, context)
    att, xd, xq = smq.DeviceBuffer(qd * 4), smq.DeviceBuffer(nb * 4), smq.DeviceBuffer(nb * 32)
    pos_dev = dev(np.array([0], np.int32))

    def run(pos, dev_pos=None):
        smq.attention_q8(qb, kb, vb, att, 1, shape, xd, xq, 0 if dev_pos else pos, dev_pos)

    graph = smq.capture(lambda: run(0, pos_dev))
    side = torch.cuda.Stream()
    for pos in positions:
        want = attend_expect(orc, q, keys, values, heads, kv_heads, hd, window, pos, 1)
        _, wd, wq = orc.quantize_q8(want)

        def check(what):
            smq.numeric_check()
            assert_same_f32(att.download(np.float32).reshape(1, qd), want, what)
            assert_same_f32(xd.download(np.float32).reshape(1, nb), wd.reshape(1, nb), what + " scales")
            assert np.array_equal(xq.download(np.int8).reshape(1, nb * 32), wq.reshape(1, nb * 32)), what
            att.upload(np.zeros(qd, np.float32))
            smq.synchronize()

        run(pos)
        check("eager")
        pos_dev.upload(np.array([pos], np.int32))
        smq.synchronize()
        graph.launch()
        check("graph")
        smq.load().smq_set_stream(side.cuda_stream)
        try:
            run(pos)
            smq.synchronize()
        finally:
            smq.load().smq_set_stream(None)
        check("another stream")
    graph.destroy()


@pytest.mark.parametrize("heads,kv_heads,hd", [(12, 2, 128), (14, 2, 64)])
def test_graphs_own_their_scores(orc, heads, kv_heads, hd):
    """Two graphs of attention on two streams at once, replayed many times beside eager calls."""
    context, pos = 1024, 1000
    qd, kd = heads * hd, kv_heads * hd
    shape = smq.attn_shape(heads, kv_heads, hd, hd // 2, 0, context)
    sets = []
    for i in range(3):
        q = synth.normal(61 + i, qd).reshape(1, qd)
        k = synth.normal(64 + i, context * kd).reshape(context, kd)
        v = synth.normal(67 + i, context * kd).reshape(context, kd)
        sets.append((dev(q), dev(k), dev(v), smq.DeviceBuffer(qd * 4),
                     attend_expect(orc, q, k, v, heads, kv_heads, hd, 0, pos, 1)))

    def run(i):
        smq.attention(sets[i][0], sets[i][1], sets[i][2], sets[i][3], 1, shape, pos)

    graphs = [smq.capture(lambda i=i: run(i)) for i in range(2)]
    side = torch.cuda.Stream()
    for _ in range(20):
        graphs[0].launch()
        run(2)
        smq.load().smq_set_stream(side.cuda_stream)
        try:
            graphs[1].launch()
        finally:
            smq.load().smq_set_stream(None)
    side.synchronize()
    smq.synchronize()
    for s in sets:
        assert_same_f32(s[3].download(np.float32).reshape(1, qd), s[4], "att")
    for g in graphs:
        g.destroy()
