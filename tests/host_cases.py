"""Cases of tests/test_host.py, each in a process of its own: host_cases.py FAKE_HIP_LIBRARY CASE. The library's host code
runs on the recording runtime of tests/fake_hip.cpp; nothing here needs a GPU."""
import ctypes
import os
import sys
import threading

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
fake = smq = None
vp = ctypes.c_void_p


class Shape(ctypes.Structure):
    _fields_ = [(n, ctypes.c_uint32) for n in ("heads", "kv_heads", "head_dim", "rotary_pairs", "window", "context")]


def load(path):
    global fake, smq
    fake = ctypes.CDLL(path, mode=ctypes.RTLD_GLOBAL)
    smq = ctypes.CDLL(os.path.join(ROOT, "smolmoe-c99_amd", "libsmq_gfx950.so"))
    for lib, names in ((fake, ("fake_log", "fake_errors")), (smq, ("smq_last_error",))):
        for n in names:
            getattr(lib, n).restype = ctypes.c_char_p
    for n in ("smq_malloc", "smq_capture_end", "smq_stream"):
        getattr(smq, n).restype = vp
    smq.smq_malloc.argtypes = [ctypes.c_size_t]
    smq.smq_set_stream.argtypes = smq.smq_graph_launch.argtypes = smq.smq_graph_destroy.argtypes = [vp]
    smq.smq_free.argtypes = [vp]
    fake.fake_fail_size.argtypes = [ctypes.c_size_t]
    fake.fake_allocations.restype = fake.fake_frees.restype = ctypes.c_uint64
    u32 = ctypes.c_uint32
    smq.smq_attention.argtypes = [vp, vp, vp, vp, u32, vp, u32, vp]
    smq.smq_attention_rope_q8.argtypes = [vp] * 3 + [vp] + [vp] * 5 + [u32] + [vp] * 3
    smq.smq_quantize_q5_rows.argtypes = [vp, u32, u32, vp]
    smq.smq_matmul.argtypes = [vp, u32, vp, vp, u32]


def init():
    assert smq.smq_init(0) == 0, smq.smq_last_error()


def log():
    return [line.split() for line in fake.fake_log().decode().splitlines()]


def kernels():
    return [w[0] for w in log()]


def errors():
    return fake.fake_errors().decode()


def stream():
    s = vp()
    assert fake.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
    return s.value


def on_thread(f):
    out = []
    t = threading.Thread(target=lambda: out.append(f()))
    t.start()
    t.join()
    return out[0]


class Attention:
    """One token's attention (ntok: up to 512) with buffers of its own."""

    def __init__(self, hd, heads=4, kv=2, context=2048, window=0):
        self.shape = Shape(heads, kv, hd, hd // 2, window, context)
        self.heads, self.hd, self.kvd, self.context = heads, hd, kv * hd, context
        self.cache = [smq.smq_malloc(context * self.kvd * 4) for _ in range(2)]
        self.pos = smq.smq_malloc(4)
        self.rows = [smq.smq_malloc(512 * heads * hd * 4) for _ in range(2)]

    def __call__(self, pos=1000, ntok=1, pos_dev=False):
        q, att = self.rows
        return smq.smq_attention(q, *self.cache, att, ntok, ctypes.byref(self.shape), pos, self.pos if pos_dev else None)


class RopeAttention(Attention):
    def __init__(self, hd, **kw):
        super().__init__(hd, **kw)
        n = self.heads * hd
        self.b = [smq.smq_malloc(n * 4), smq.smq_malloc(self.kvd * 4), smq.smq_malloc(self.kvd * 4)]
        self.tables = [smq.smq_malloc(self.context * hd * 2) for _ in range(2)]
        self.out = [smq.smq_malloc(n * 4), smq.smq_malloc(n // 32 * 4), smq.smq_malloc(n)]

    def __call__(self, pos=1000, pos_dev=False):
        return smq.smq_attention_rope_q8(*self.b, ctypes.byref(self.shape), *self.tables, *self.cache, self.out[0], pos,
                                         self.pos if pos_dev else None, self.out[1], self.out[2])


def capture(f):
    assert smq.smq_capture_begin() == 0, smq.smq_last_error()
    assert f() == 0, smq.smq_last_error()
    g = smq.smq_capture_end()
    assert g, smq.smq_last_error()
    return g


def both_at_once(graphs, side):
    """The graphs on two streams without an order between them."""
    assert smq.smq_graph_launch(graphs[0]) == 0
    smq.smq_set_stream(side)
    assert smq.smq_graph_launch(graphs[1]) == 0
    smq.smq_set_stream(None)


def nested_capture():
    """A begin inside an open capture, of the same thread or another, is refused and changes nothing: the graph still
    owns the workspace that it recorded."""
    for other in (False, True):
        init()
        att = Attention(128)
        assert smq.smq_capture_begin() == 0
        assert att() == 0
        assert (on_thread(smq.smq_capture_begin) if other else smq.smq_capture_begin()) != 0
        assert fake.hipGetLastError() == 0  # nothing for the next launch to find
        first = smq.smq_capture_end()
        assert first
        second = capture(att)
        fake.fake_clear()
        both_at_once((first, second), stream())
        assert len({w[8] for w in log()}) == 2, fake.fake_log().decode()
        smq.smq_graph_destroy(second)
        assert smq.smq_graph_launch(first) == 0
        assert errors() == "", errors()
        smq.smq_graph_destroy(first)
        smq.smq_shutdown()


def failed_captures():
    """A capture that fails (a call that it does not allow) or is ended on the wrong stream leaves the next ones whole."""
    init()
    att, side = Attention(128), stream()
    assert smq.smq_capture_begin() == 0 and att() == 0
    assert smq.smq_malloc(64) is None
    assert smq.smq_capture_end() is None
    fake.hipGetLastError()
    assert smq.smq_capture_begin() == 0 and att() == 0
    smq.smq_set_stream(side)
    assert smq.smq_capture_end() is None  # the library's stream is still capturing
    fake.hipGetLastError()
    smq.smq_set_stream(None)
    assert smq.smq_capture_begin() != 0
    first = smq.smq_capture_end()
    assert first
    second = capture(att)
    fake.fake_clear()
    both_at_once((first, second), side)
    assert errors() == "", errors()


def destroyed_handle():
    """A graph made while another is destroyed may get its handle, and keeps its own workspace."""
    init()
    att, made = Attention(128), []
    first = capture(att)
    hook = ctypes.CFUNCTYPE(None)(lambda: made.append(capture(att)))
    fake.fake_on_exec_destroy(hook)
    smq.smq_graph_destroy(first)
    assert made == [first]  # the handle again
    capture(att)
    assert smq.smq_graph_launch(made[0]) == 0
    assert errors() == "", errors()


def stream_read_once():
    """A stream set by another thread during a call does not move the rest of the call, nor the workspace with it."""
    init()
    own, side = smq.smq_stream(), stream()
    hook = ctypes.CFUNCTYPE(None)(lambda: smq.smq_set_stream(side))
    for att, ntok in ((Attention(128), 1), (Attention(128), 200), (Attention(48), 200)):
        smq.smq_set_stream(None)
        fake.fake_clear()
        fake.fake_on_is_capturing(hook)
        assert att(ntok=ntok) == 0
        assert smq.smq_stream() == side and log()
        assert {int(w[6], 16) for w in log()} == {own}, fake.fake_log().decode()


def two_launches():
    names = kernels()
    return any("k_attend_scores" in n for n in names) and any("k_attend_values" in n for n in names)


def scores_by_stream():
    """Decode attention in graphs, beside eager calls and on other streams: no two uses of a workspace without an order,
    and two launches wherever the workspace can be had."""
    for make in (lambda: Attention(64), lambda: RopeAttention(64), lambda: Attention(128)):
        init()
        att, own, side, third = make(), smq.smq_stream(), stream(), stream()
        split = att.hd != 64  # on the library's own stream only
        graphs = [capture(lambda: att(pos_dev=True)) for _ in range(2)]
        fake.fake_clear()
        both_at_once(graphs, side)
        assert att() == 0  # eager, beside both
        assert two_launches() and errors() == "", errors()

        def call(s, expected):
            fake.fake_clear()
            smq.smq_set_stream(s)
            assert att() == 0
            assert two_launches() == expected and errors() == "", fake.fake_log().decode() + errors()

        fourth = stream()
        for s in (side, None, third, side, None, third):  # a workspace for each of three streams, without a wait
            call(s, not split or s is None)
        call(fourth, False)  # the launch that needs none
        call(side, not split)
        assert smq.smq_synchronize() == 0
        call(fourth, not split)  # the other's use is over
        call(side, False)
        smq.smq_free(smq.smq_malloc(64))  # waits for the device
        for s in (side, fourth, None):
            call(s, not split or s is None)
        call(third, False)

        for s in (side, own):  # a capture that the program opened itself
            smq.smq_set_stream(s)
            assert fake.hipStreamBeginCapture(vp(s), 1) == 0
            assert att() == 0
            graph, exe = vp(), vp()
            assert fake.hipStreamEndCapture(vp(s), ctypes.byref(graph)) == 0
            assert fake.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
            smq.smq_set_stream(None)
            assert att() == 0
            fake.fake_clear()
            assert fake.hipGraphLaunch(exe, vp(third)) == 0
            assert not two_launches() and errors() == "", errors()
        for g in graphs:
            smq.smq_graph_destroy(g)
        smq.smq_shutdown()


def no_memory():
    """Without memory for a score workspace the library starts, captures and computes with the kernels that need none."""
    fake.fake_fail_size(128 << 20)
    init()
    for hd, ntok in ((128, 1), (64, 1), (128, 200), (64, 200)):
        att = Attention(hd)
        fake.fake_clear()
        assert att(ntok=ntok) == 0, smq.smq_last_error()
        assert log() and not any("k_ap_" in n for n in kernels()) and errors() == ""
    fake.fake_fail_size(16 << 20)
    graphs = [capture(Attention(hd)) for hd in (128, 64, 128, 64)]
    for g in graphs:
        fake.fake_clear()
        assert smq.smq_graph_launch(g) == 0
        assert log() and errors() == "", errors()
        smq.smq_graph_destroy(g)


def captures_again():
    """A program that captures its decode step again after each prompt allocates and frees nothing, and a workspace is
    not handed on while a replay may be using it."""
    init()
    att, side = Attention(128), stream()
    before = fake.fake_allocations(), fake.fake_frees()
    for _ in range(8):
        g = capture(att)
        assert smq.smq_graph_launch(g) == 0
        assert smq.smq_synchronize() == 0
        smq.smq_graph_destroy(g)
    assert (fake.fake_allocations(), fake.fake_frees()) == before
    for launched_on in (None, side):  # destroyed behind a replay that nobody waited for
        first = capture(att)
        smq.smq_set_stream(launched_on)
        assert smq.smq_graph_launch(first) == 0
        smq.smq_set_stream(None)
        smq.smq_graph_destroy(first)
        second = capture(att)
        smq.smq_set_stream(stream())
        assert smq.smq_graph_launch(second) == 0
        smq.smq_set_stream(None)
        smq.smq_graph_destroy(second)
    assert errors() == "", errors()
    graphs = [capture(att) for _ in range(12)]  # no more kept than a few
    for g in graphs:
        smq.smq_graph_destroy(g)
    assert fake.fake_allocations() - fake.fake_frees() - (before[0] - before[1]) <= 4
    kept = [capture(att) for _ in range(2)]  # across a shutdown: freed with their graph
    smq.smq_shutdown()
    for g in kept:
        smq.smq_graph_destroy(g)
    assert errors() == "", errors()


def tile_routes():
    """Every shape of the GPU test of the attention tiles reaches them, and none in a capture or on another stream."""
    sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
    from test_gpu_attend_tiles import CASES as SHAPES
    init()
    side = stream()
    for heads, kv, hd, window, context, ntok, pos0 in SHAPES:
        att = Attention(hd, heads, kv, context, window)
        for s in (None, side):
            smq.smq_set_stream(s)
            fake.fake_clear()
            assert att(pos0, ntok) == 0, smq.smq_last_error()
            names = kernels()
            tiles = [any(k in n for n in names) for k in ("k_ap_scores", "k_ap_softmax", "k_ap_values")]
            assert tiles == [s is None] * 3, (heads, kv, hd, window, context, ntok, pos0, names)
        smq.smq_set_stream(None)
        fake.fake_clear()
        assert smq.smq_graph_launch(capture(lambda: att(pos0, ntok))) == 0
        assert not any("k_ap" in n for n in kernels())


def attention_routes():
    """Both sides of the lines between the prefill kernels and between the decode kernels."""
    init()
    prefill = [  # heads, kv_heads, hd, window, context, ntok, pos0, kernel
        (14, 2, 64, 0, 1024, 512, 0, "k_ap_"), (14, 2, 64, 0, 1024, 2, 256, "k_attend_group"),
        (14, 2, 64, 0, 1024, 2, 1000, "k_ap_"), (9, 3, 64, 512, 964, 17, 564, "k_attend_group"),
        (9, 3, 64, 0, 644, 16, 572, "k_attend_group"), (32, 8, 64, 512, 853, 61, 718, "k_attend_group"),
        (32, 8, 64, 0, 363, 89, 202, "k_ap_"), (14, 2, 64, 128, 2002, 22, 331, "k_attend_rows"),
        (9, 3, 64, 128, 5078, 40, 3276, "k_attend_rows"), (14, 2, 64, 0, 2002, 16, 1000, "k_attend_rows"),
        (14, 2, 64, 0, 4000, 16, 3800, "k_ap_"), (12, 2, 128, 0, 3100, 8, 3000, "k_ap_"),
        (12, 2, 128, 0, 600, 4, 500, "k_attendE"), (16, 2, 36, 0, 3100, 64, 3000, "k_attendE"),
    ]
    decode = [  # heads, kv_heads, hd, window, context, pos, kernel
        (14, 2, 64, 0, 2048, 5, "k_attend_values"), (12, 2, 128, 0, 2048, 150, "k_attendE"),
        (12, 2, 128, 0, 2048, 151, "k_attend_values"), (12, 2, 128, 100, 2048, 1000, "k_attendE"),
        (9, 3, 32, 0, 2048, 246, "k_attendE"), (9, 3, 32, 0, 2048, 247, "k_attend_values"),
        (17, 1, 128, 0, 2048, 1000, "k_attendE"), (17, 1, 64, 0, 2048, 1000, "k_attend_rows"),
        (9, 3, 48, 0, 2048, 1000, "k_attendE"),
    ]
    for heads, kv, hd, window, context, *rest in prefill + [(*d[:5], 1, *d[5:]) for d in decode]:
        ntok, pos, want = rest
        att = Attention(hd, heads, kv, context, window)
        fake.fake_clear()
        assert att(pos, ntok) == 0, smq.smq_last_error()
        assert want in kernels()[-1], (heads, kv, hd, window, context, rest, kernels())


def matmul_routes():
    """Both sides of the lines between the kernels of 2-16 tokens (256 CUs)."""
    sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
    from smq_pkg import smq as package
    QMat, Item = package._QMat, package._MatItem
    init()
    w, x, y = (smq.smq_malloc(1 << 30) for _ in range(3))
    four, wide = "k_gemm_xmILb%dELb0ELi4E", "k_gemm_xmILb%dELb0ELi1E"
    dot8, dot16, few = "k_gemm_exactILb%dELb0ELi8E", "k_gemm_exactILb%dELb0ELi16E", "k_gemv_fewILb%d"
    table = [  # rows, cols, ntok, Q8, Q5
        (4096, 896, 12, dot8, dot8), (4128, 896, 12, four, four), (4864, 4864, 11, four, four),
        (4864, 384, 16, dot8, dot8), (4864, 448, 16, four, four), (5120, 384, 16, four, four),
        (14304, 576, 16, four, four), (14336, 576, 16, wide, wide), (24576, 576, 9, wide, wide), (24576, 896, 9, four, four),
        (65536, 896, 16, wide, wide), (65504, 896, 16, four, four), (16384, 896, 8, dot8, dot8),
        (2048, 448, 4, few, few), (2688, 448, 4, dot8, dot8), (16384, 1536, 4, few, dot8), (16400, 1536, 4, dot8, dot8),
        (12288, 1536, 3, few, few), (4096, 896, 2, few, few), (4128, 896, 2, few, dot8), (1024, 1536, 12, few, few),
        (1024, 896, 16, dot8, dot8), (1024, 1984, 16, few, few),
    ]
    for rows, cols, ntok, *wants in table:
        for q5, want in enumerate(wants):
            nb = (cols + 31) // 32
            m = QMat(w, rows, cols, nb, package.DTYPE_Q5 if q5 else package.DTYPE_Q8, nb * (22 if q5 else 36))
            item = Item(ctypes.pointer(m), None, y, 0)
            fake.fake_clear()
            assert smq.smq_matmul(ctypes.byref(item), 1, x, x, ntok) == 0, smq.smq_last_error()
            assert want % q5 in kernels()[0], (rows, cols, ntok, q5, kernels())


def conversion_limits():
    """Q5 conversion: both sides of the line between one and two rounds, and the most blocks (addresses only)."""
    init()
    x, out = smq.smq_malloc(18 << 30), smq.smq_malloc(95 << 30)
    for rows, kernel, grid in ((1, "Lj1E", 1), (28000, "Lj1E", 2334), (28001, "Lj2E", 1167),
                               (2**32 - 1, "Lj2E", (2**32 - 1 + 23) // 24)):
        fake.fake_clear()
        assert smq.smq_quantize_q5_rows(x, rows, 1, out) == 0, smq.smq_last_error()
        assert kernel in kernels()[0] and int(log()[0][2]) == grid, log()
    fake.fake_clear()
    assert smq.smq_quantize_q5_rows(x, 2**31, 65, out) != 0 and not log()  # past both allocations


def capture_with_an_exception():
    """The binding's capture of a function that raises leaves neither a graph nor its workspace behind."""
    sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
    from smq_pkg import smq as package
    init()
    package.load()
    att, before = Attention(128), fake.fake_allocations()

    def broken():
        assert att() == 0
        raise KeyError("in the middle")

    for _ in range(5):
        try:
            package.capture(broken)
        except KeyError:
            continue
        raise AssertionError("no exception")
    assert fake.fake_allocations() == before and errors() == "", errors()
    package.capture(lambda: att()).destroy()


CASES = [f for f in (nested_capture, failed_captures, destroyed_handle, stream_read_once, scores_by_stream, no_memory,
                     captures_again, capture_with_an_exception, tile_routes, attention_routes, matmul_routes, conversion_limits)]

if __name__ == "__main__":
    load(sys.argv[1])
    {f.__name__: f for f in CASES}[sys.argv[2]]()
    print("ok")
