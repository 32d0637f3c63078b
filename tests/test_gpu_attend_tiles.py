"""Prefill attention in 16-row tiles (csrc/smq_attend.hip) against the oracle's attend_f32, bit for bit, and
against the kernels that need no workspace (the route of a captured call)."""
import numpy as np
import pytest

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


CASES = [  # heads, kv_heads, hd, window, context, ntok, pos0 (each past the rule that chooses the tiles)
    (14, 2, 64, 0, 1100, 83, 1010),     # seven heads per group: tiles that straddle tokens, a partial last tile
    (14, 2, 64, 0, 1024, 5, 1019),      # a context the grouped kernel serves, up to its end
    (12, 2, 128, 0, 700, 11, 645),      # head_dim 128, past a chunk of positions
    (4, 4, 128, 0, 300, 97, 0),         # one head per group: 16 tokens per tile, from position 0
    (8, 4, 16, 0, 200, 101, 70),        # head_dim 16: one group of the dot, half of it padded
    (9, 3, 48, 0, 600, 70, 250),        # head_dim 48
    (16, 2, 80, 0, 300, 33, 255),       # head_dim 80: five column tiles
    (8, 8, 96, 0, 600, 40, 500),        # head_dim 96
    (5, 1, 104, 0, 370, 55, 256),       # head_dim 104: half a column tile
    (2, 1, 256, 0, 300, 97, 150),       # head_dim 256: the largest
    (9, 3, 24, 0, 400, 101, 280),       # head_dim 24
    (8, 2, 8, 0, 200, 103, 3),          # head_dim 8: the smallest
    (32, 1, 32, 0, 200, 41, 150),       # more heads in a group than rows in a tile
    (14, 2, 64, 100, 1500, 37, 1400),   # a sliding window: tile bases in the middle of the cache
    (8, 2, 32, 5, 200, 200, 0),         # a window smaller than a tile, every position of the context
    (64, 64, 16, 0, 16384, 20, 16360),  # the longest context, two slabs of the workspace
]


@pytest.mark.parametrize("heads,kv_heads,hd,window,context,ntok,pos0", CASES)
def test_attend_tiles(orc, heads, kv_heads, hd, window, context, ntok, pos0):
    say("attend tiles", heads, kv_heads, hd, window, context, ntok, pos0)
    qd, kd = heads * hd, kv_heads * hd
    nb = (qd + 31) // 32
    q = synth.normal(41, ntok * qd, 2.0).reshape(ntok, qd)
    keys = synth.normal(42, context * kd).reshape(context, kd)
    values = synth.normal(43, context * kd).reshape(context, kd)
    qb, kb, vb = dev(q), dev(keys), dev(values)
    shape = smq.attn_shape(heads, kv_heads, hd, hd // 2, window, context)

    def outputs():
        return smq.DeviceBuffer(ntok * qd * 4), smq.DeviceBuffer(ntok * nb * 4), smq.DeviceBuffer(ntok * nb * 32)

    tiles, plain = outputs(), outputs()
    smq.attention_q8(qb, kb, vb, tiles[0], ntok, shape, tiles[1], tiles[2], pos0)
    graph = smq.capture(lambda: smq.attention_q8(qb, kb, vb, plain[0], ntok, shape, plain[1], plain[2], pos0))
    graph.launch()
    smq.numeric_check()
    graph.destroy()
    att = tiles[0].download(np.float32).reshape(ntok, qd)
    assert_same_f32(att, plain[0].download(np.float32).reshape(ntok, qd), "att of the captured call")
    assert_same_f32(tiles[1].download(np.float32), plain[1].download(np.float32), "scales of the captured call")
    assert np.array_equal(tiles[2].download(np.int8), plain[2].download(np.int8))
    rows = range(ntok) if ntok * heads * (pos0 + ntok) * hd < 1 << 28 else (0, 15, 16, ntok - 1)
    for t in rows:
        want = attend_expect(orc, q[t:t + 1], keys, values, heads, kv_heads, hd, window, pos0 + t, 1)
        assert_same_f32(att[t:t + 1], want, f"att of token {t}")


def test_attend_tiles_later_rows_do_not_reach_earlier_tokens(orc):
    """A non-finite value row of a later token of the batch reaches only the tokens that see it."""
    heads, kv_heads, hd, context, ntok, pos0 = 40, 2, 64, 1100, 48, 30
    qd, kd = heads * hd, kv_heads * hd
    q = synth.normal(44, ntok * qd).reshape(ntok, qd)
    keys = synth.normal(45, context * kd).reshape(context, kd)
    values = synth.normal(46, context * kd).reshape(context, kd)
    values[pos0 + 5:] = np.inf
    keys[pos0 + 6:] = np.nan
    att = smq.DeviceBuffer(ntok * qd * 4)
    shape = smq.attn_shape(heads, kv_heads, hd, hd // 2, 0, context)
    smq.attention(dev(q), dev(keys), dev(values), att, ntok, shape, pos0)
    smq.synchronize()
    want = attend_expect(orc, q[:5], keys, values, heads, kv_heads, hd, 0, pos0, 5)
    got = att.download(np.float32).reshape(ntok, qd)
    assert_same_f32(got[:5], want, "tokens before the non-finite row")
    assert not np.isfinite(got[5:]).any()


@pytest.mark.parametrize("scale", ["spread", "tiny"])
@pytest.mark.parametrize("heads,kv_heads,hd,context,ntok,pos0", [(14, 2, 64, 1100, 20, 1010), (12, 2, 128, 700, 11, 645),
                                                                 (8, 4, 16, 200, 101, 70)])
def test_attend_tiles_small_values(orc, scale, heads, kv_heads, hd, context, ntok, pos0):
    """Weights that are subnormal or zero (a wide spread of scores); scores, values and products that are subnormal."""
    say("attend tiles", scale, heads, hd)
    qd, kd = heads * hd, kv_heads * hd
    qs, ks, vs = (30.0, 1.0, 1.0) if scale == "spread" else (1e-20, 1e-20, 3e-39)
    q = synth.normal(47, ntok * qd, qs).reshape(ntok, qd)
    keys = synth.normal(48, context * kd, ks).reshape(context, kd)
    values = synth.normal(49, context * kd, vs).reshape(context, kd)
    att = smq.DeviceBuffer(ntok * qd * 4)
    smq.attention(dev(q), dev(keys), dev(values), att, ntok, smq.attn_shape(heads, kv_heads, hd, hd // 2, 0, context), pos0)
    smq.synchronize()
    want = attend_expect(orc, q, keys, values, heads, kv_heads, hd, 0, pos0, ntok)
    assert np.isfinite(want).all() and want.any()
    assert_same_f32(att.download(np.float32).reshape(ntok, qd), want, scale)


@pytest.mark.parametrize("what", ["inf value", "inf - inf", "nan value", "nan key", "inf key", "-inf key"])
@pytest.mark.parametrize("heads,kv_heads,hd,context,ntok,pos0", [(14, 2, 64, 1400, 20, 1010), (12, 2, 128, 1400, 11, 645),
                                                                 (14, 2, 64, 1400, 1, 1300), (6, 2, 96, 1400, 1, 1300)])
def test_attend_non_finite(orc, what, heads, kv_heads, hd, context, ntok, pos0):
    """Non-finite keys and values among the positions that the rows see, in the tiles and in the long value path."""
    say("attend", what, heads, hd, ntok)
    qd, kd = heads * hd, kv_heads * hd
    q = synth.normal(57, ntok * qd).reshape(ntok, qd)
    keys = synth.normal(58, context * kd).reshape(context, kd)
    values = synth.normal(59, context * kd).reshape(context, kd)
    at = pos0 - 20
    if what.endswith("key"):
        keys[at, kd - hd + 5] = {"nan key": np.nan, "inf key": np.inf, "-inf key": -np.inf}[what]
    else:
        values[at, 3] = np.nan if what == "nan value" else np.inf
        if what == "inf - inf":
            values[at + 9, 3] = -np.inf
    att = smq.DeviceBuffer(ntok * qd * 4)
    smq.attention(dev(q), dev(keys), dev(values), att, ntok, smq.attn_shape(heads, kv_heads, hd, hd // 2, 0, context), pos0)
    smq.synchronize()
    want = attend_expect(orc, q, keys, values, heads, kv_heads, hd, 0, pos0, ntok)
    assert_same_f32(att.download(np.float32).reshape(ntok, qd), want, what)
