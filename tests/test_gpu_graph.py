"""The hot path under HIP graph capture. The library enqueues on one stream that it hands out
(iris_dev_stream), and the two hot-path operators allocate nothing on the layouts the matrix-core
kernels take directly (head_dim 128 / 256 / 512, 16-byte aligned rows), so a caller can capture a
step -- norm+rope on Q, on K, attention -- into a graph once and replay it (what a launch-bound loop
such as the 36 layers of the text encoder wants). Every replay is checked against the eager result,
with eager work and synchronisations of the program between the replays.
"""
import ctypes as C

import numpy as np
import pytest

import workloads as W
from gpu_harness import Dev, ptr_add

pytestmark = pytest.mark.gpu
_vp = C.c_void_p


class Graphs:
    def __init__(self):
        self.rt = C.CDLL("libamdhip64.so")
        self.rt.hipStreamBeginCapture.argtypes = [_vp, C.c_int]
        self.rt.hipStreamEndCapture.argtypes = [_vp, C.POINTER(_vp)]
        self.rt.hipGraphInstantiate.argtypes = [C.POINTER(_vp), _vp, _vp, _vp, C.c_size_t]
        self.rt.hipGraphLaunch.argtypes = [_vp, _vp]
        self.rt.hipGraphExecDestroy.argtypes = [_vp]
        self.rt.hipGraphDestroy.argtypes = [_vp]
        self.rt.hipGraphGetNodes.argtypes = [_vp, _vp, C.POINTER(C.c_size_t)]
        self.rt.hipStreamCreate.argtypes = [C.POINTER(_vp)]
        self.rt.hipStreamSynchronize.argtypes = [_vp]
        self.rt.hipStreamDestroy.argtypes = [_vp]

    def capture(self, stream, fn):
        assert self.rt.hipStreamBeginCapture(stream, 0) == 0          # hipStreamCaptureModeGlobal
        fn()
        graph, run = _vp(), _vp()
        assert self.rt.hipStreamEndCapture(stream, C.byref(graph)) == 0 and graph
        nodes = C.c_size_t()
        assert self.rt.hipGraphGetNodes(graph, None, C.byref(nodes)) == 0
        self.nodes = nodes.value
        assert self.rt.hipGraphInstantiate(C.byref(run), graph, None, None, 0) == 0
        self.rt.hipGraphDestroy(graph)
        return run


@pytest.mark.parametrize("maker", [W.c1, W.c4, lambda: W.c2(shrink=4), W.c2], ids=["c1", "c4", "c2-shrunk", "c2-two-size-grid"])
def test_step_replayed_from_a_graph_equals_the_eager_step(maker):
    case = maker()
    dev, g = Dev(), Graphs()
    lib, stream = dev.lib, _vp(dev.lib.iris_dev_stream())
    seq, ldi, qd, kd = case["seq"], case["ldi"], case["q_dim"], case["kv_dim"]
    rows, out = dev.put(case["buf"]), dev.alloc(seq * case["ldo"] * 2)
    wq, wk, cos, sin = dev.put(case["wq"]), dev.put(case["wk"]), dev.put(case["cos"]), dev.put(case["sin"])
    mask = dev.put(np.ascontiguousarray(case["key_mask"], np.int32)) if case["key_mask"] is not None else None

    def step():
        lib.iris_dev_head_norm_rope(rows, ldi, wq, cos, sin, seq, case["heads"], 128, case["eps"], case["split_half"])
        lib.iris_dev_head_norm_rope(ptr_add(rows, 2 * qd), ldi, wk, cos, sin, seq, case["kv_heads"], 128, case["eps"], case["split_half"])
        lib.iris_dev_attention(out, case["ldo"], rows, ptr_add(rows, 2 * qd), ptr_add(rows, 2 * (qd + kd)), ldi, seq, seq,
                               case["heads"], case["kv_heads"], 128, case["scale"], int(case["causal"]), mask)

    step()                                              # eager (also the first launch of each kernel: attributes are set here)
    dev.check()
    want = dev.get(out, (seq, case["ldo"]), np.uint16)
    assert want.any()
    run = g.capture(stream, step)
    dev.check()
    host = np.ascontiguousarray(case["buf"])
    for replay in range(4):
        # eager work of the program between the replays: the rows are normalised in place, so they are uploaded again,
        # and the output is overwritten with a pattern
        lib.iris_dev_upload(rows, host.ctypes.data_as(_vp), host.nbytes)
        junk = np.full((seq, case["ldo"]), 0x7fc0 + replay, np.uint16)
        lib.iris_dev_upload(out, junk.ctypes.data_as(_vp), junk.nbytes)
        assert g.rt.hipGraphLaunch(run, stream) == 0
        lib.iris_dev_sync()
        dev.check()
        got = dev.get(out, (seq, case["ldo"]), np.uint16)
        assert np.array_equal(got, want), f"replay {replay} differs from the eager step"
    g.rt.hipGraphExecDestroy(run)
    dev.free_all()


def test_a_layout_that_needs_scratch_is_refused_during_capture_until_the_scratch_exists():
    """head_dim 64 runs on the matrix cores through a padded private copy of q | k | v. Growing that copy means
    synchronise + free + allocate, which would invalidate a capture: inside a capture the call is refused (error
    reported, nothing enqueued, the capture stays valid); after one call outside, the same call is captured and
    replays to the eager result."""
    import oracle as O
    dev, g = Dev(), Graphs()
    lib, stream = dev.lib, _vp(dev.lib.iris_dev_stream())
    rng = np.random.default_rng(3)
    seq, heads, hd = 30000, 2, 64          # a 46 MB copy: larger than anything another test has left in the scratch
    buf = O.f32_to_bf16(rng.standard_normal((seq, 3 * heads * hd)).astype(np.float32))
    rows, out = dev.put(buf), dev.alloc(seq * heads * hd * 2)
    args = (out, heads * hd, rows, ptr_add(rows, 2 * heads * hd), ptr_add(rows, 4 * heads * hd), 3 * heads * hd, seq, seq, heads, heads, hd,
            0.125, 0, None)
    assert g.rt.hipStreamBeginCapture(stream, 0) == 0
    lib.iris_dev_attention(*args)
    refused = lib.iris_dev_last_error()
    graph = _vp()
    assert g.rt.hipStreamEndCapture(stream, C.byref(graph)) == 0, "the refused call must leave the capture valid"
    if graph:
        g.rt.hipGraphDestroy(graph)
    assert refused == -1
    lib.iris_dev_attention(*args)                                   # outside: allocates the scratch
    dev.check()
    assert dev.dev.last_kernel() == "fa_hd128_packed"
    want = dev.get(out, (seq, heads * hd), np.uint16)
    assert want.any()
    run = g.capture(stream, lambda: lib.iris_dev_attention(*args))
    dev.check()
    for replay in range(2):
        junk = np.full((seq, heads * hd), 0x7fc0 + replay, np.uint16)
        lib.iris_dev_upload(out, junk.ctypes.data_as(_vp), junk.nbytes)
        assert g.rt.hipGraphLaunch(run, stream) == 0
        lib.iris_dev_sync()
        assert np.array_equal(dev.get(out, (seq, heads * hd), np.uint16), want)
    g.rt.hipGraphExecDestroy(run)
    dev.free_all()


def test_double_stream_step_replayed_from_a_graph():
    """The joint block's step with the one-launch norm of both streams (iris_dev_head_norm_rope_qk_streams: text rows
    and image rows with their own weight pairs) and attention, captured once and replayed: every replay equals the
    eager step bit for bit."""
    case = W.c2(shrink=4)
    dev, g = Dev(), Graphs()
    lib, stream = dev.lib, _vp(dev.lib.iris_dev_stream())
    seq, ldi, qd, kd = case["seq"], case["ldi"], case["q_dim"], case["kv_dim"]
    txt = 512 // 4
    rows, out = dev.put(case["buf"]), dev.alloc(seq * case["ldo"] * 2)
    wq, wk, cos, sin = dev.put(case["wq"]), dev.put(case["wk"]), dev.put(case["cos"]), dev.put(case["sin"])
    wq2, wk2 = dev.put(case["wq"][::-1].copy()), dev.put(case["wk"][::-1].copy())

    def step():
        lib.iris_dev_head_norm_rope_qk_streams(rows, ptr_add(rows, 2 * qd), ldi, wq, wk, wq2, wk2, txt, cos, sin, seq, case["heads"],
                                               case["kv_heads"], 128, case["eps"], 0)
        lib.iris_dev_attention(out, case["ldo"], rows, ptr_add(rows, 2 * qd), ptr_add(rows, 2 * (qd + kd)), ldi, seq, seq,
                               case["heads"], case["kv_heads"], 128, case["scale"], 0, None)

    step()
    dev.check()
    want = dev.get(out, (seq, case["ldo"]), np.uint16)
    assert want.any()
    run = g.capture(stream, step)
    dev.check()
    host = np.ascontiguousarray(case["buf"])
    for replay in range(3):
        lib.iris_dev_upload(rows, host.ctypes.data_as(_vp), host.nbytes)
        junk = np.full((seq, case["ldo"]), 0x7fc0 + replay, np.uint16)
        lib.iris_dev_upload(out, junk.ctypes.data_as(_vp), junk.nbytes)
        assert g.rt.hipGraphLaunch(run, stream) == 0
        lib.iris_dev_sync()
        dev.check()
        assert np.array_equal(dev.get(out, (seq, case["ldo"]), np.uint16), want), f"replay {replay} differs from the eager step"
    g.rt.hipGraphExecDestroy(run)
    dev.free_all()


@pytest.mark.parametrize("causal_and_masked", [False, True], ids=["plain", "causal-masked"])
def test_head_dim_512_attention_with_key_ranges_replayed_from_a_graph(causal_and_masked):
    """The VAE's attention call at 4096 tokens: two launches (key ranges, then their merge through private scratch), and
    with a key mask a third in front that packs the mask into the same scratch. Once the scratch exists the call is
    captured; every replay, with eager calls of another size between them that overwrite the same scratch, equals
    the eager result."""
    import oracle as O
    dev, g = Dev(), Graphs()
    lib, stream = dev.lib, _vp(dev.lib.iris_dev_stream())
    rng = np.random.default_rng(5)
    seq, hd = 4096, 512
    buf = O.f32_to_bf16(rng.standard_normal((seq, 3 * hd)).astype(np.float32))
    rows, out, other = dev.put(buf), dev.alloc(seq * hd * 2), dev.alloc(seq * hd * 2)
    scale = float(1 / np.sqrt(hd))
    causal = int(causal_and_masked)
    mask = dev.put((rng.random(seq) < 0.7).astype(np.int32)) if causal_and_masked else None
    args = (out, hd, rows, ptr_add(rows, 2 * hd), ptr_add(rows, 4 * hd), 3 * hd, seq, seq, 1, 1, hd, scale, causal, mask)
    small = (other, hd, rows, ptr_add(rows, 2 * hd), ptr_add(rows, 4 * hd), 3 * hd, 1000, 1000, 1, 1, hd, scale, causal, mask)
    lib.iris_dev_attention(*args)                                   # outside: the scratch is sized
    dev.check()
    assert dev.dev.last_kernel() == "fa_hd512"
    want = dev.get(out, (seq, hd), np.uint16)
    run = g.capture(stream, lambda: lib.iris_dev_attention(*args))
    dev.check()
    for replay in range(3):
        junk = np.full((seq, hd), 0x7fc0 + replay, np.uint16)
        lib.iris_dev_upload(out, junk.ctypes.data_as(_vp), junk.nbytes)
        lib.iris_dev_attention(*small)                              # eager work on the same scratch between the replays
        assert g.rt.hipGraphLaunch(run, stream) == 0
        lib.iris_dev_sync()
        assert np.array_equal(dev.get(out, (seq, hd), np.uint16), want), f"replay {replay}"
    g.rt.hipGraphExecDestroy(run)
    dev.free_all()


@pytest.mark.parametrize("bf16", [False, True])
def test_captured_linear_layer_uses_no_shared_memory(bf16):
    """300 x 4096 -> 640 is cut into ranges of K, whose partial sums share the library's workspace in stream order. Captured,
    the layer is one kernel on its own operands, so its replays on another stream and eager layers that use the
    workspace meanwhile both give their results. The replay sums K in another order: f32 rounding apart from the eager call."""
    import oracle as O
    dev, g = Dev(), Graphs()
    lib, stream = dev.lib, _vp(dev.lib.iris_dev_stream())
    rows, k, out = 300, 4096, 640
    plan = (C.c_int * 2)()
    lib.iris_hip_linear_plan(rows, k, out, 2 if bf16 else 4, plan)
    assert plan[0] == 4 and plan[1] > 1
    rng = np.random.default_rng(8)
    x = O.f32_to_bf16(rng.standard_normal((rows, k)).astype(np.float32))
    weights = [O.f32_to_bf16((rng.standard_normal((out, k)) * 0.05).astype(np.float32)) for _ in range(2)]
    want = [O.bf16_to_f32(x).astype(np.float64) @ O.bf16_to_f32(w).astype(np.float64).T for w in weights]
    dx, (w1, w2) = dev.put(x), [dev.put(w) for w in weights]
    size = 2 if bf16 else 4
    captured, eager = dev.alloc(rows * out * size), dev.alloc(rows * out * size)
    layer = lib.iris_dev_linear_bf16 if bf16 else lib.iris_dev_linear_f32

    def check(ptr, w):
        got = dev.get(ptr, (rows, out), np.uint16 if bf16 else np.float32)
        got = O.bf16_to_f32(got) if bf16 else got
        # f32 sums of 4096 products of size 0.05, and the rounding to bf16
        assert (np.abs(got - want[w]) <= 2e-5 * np.sqrt(k) * 0.05 + (np.abs(want[w]) * 2.0 ** -8 * 1.01 if bf16 else 0.0)).all()

    layer(eager, dx, w2, rows, k, out)
    run = g.capture(stream, lambda: layer(captured, dx, w1, rows, k, out))
    assert g.nodes == 1
    dev.check()
    lib.iris_dev_sync()
    other = _vp()
    assert g.rt.hipStreamCreate(C.byref(other)) == 0
    junk = np.full(rows * out * size // 2, 0x7fc0, np.uint16)
    for replay in range(4):
        for p in (captured, eager):
            lib.iris_dev_upload(p, junk.ctypes.data_as(_vp), junk.nbytes)
        for _ in range(8):
            assert g.rt.hipGraphLaunch(run, other) == 0
            layer(eager, dx, w2, rows, k, out)
        assert g.rt.hipStreamSynchronize(other) == 0
        lib.iris_dev_sync()
        dev.check()
        check(captured, 0)
        check(eager, 1)
    g.rt.hipGraphExecDestroy(run)
    g.rt.hipStreamDestroy(other)
    dev.free_all()


def test_captured_convolution_uses_no_shared_memory():
    """64 x 69, 512 -> 256: the last round of tiles is cut into ranges of input channels, whose sums share the workspace of the linear
    layers in stream order. Captured, the convolution is one kernel on its own operands, so its replays on another stream give their
    result beside eager convolutions and layers that use the workspace one after the other, and so do those. The replay sums the
    channels in another order: f32 rounding apart from the eager call."""
    import oracle as O
    from test_gpu_conv_direct import conv_float64
    dev, g = Dev(), Graphs()
    lib, stream = dev.lib, _vp(dev.lib.iris_dev_stream())
    h, w, cin, cout = 64, 69, 512, 256
    rows, k, out = 300, 4096, 640
    assert lib.iris_hip_conv2d_cut(h, w, cin, cout) == 1
    plan = (C.c_int * 2)()
    lib.iris_hip_linear_plan(rows, k, out, 4, plan)
    assert plan[0] == 4 and plan[1] > 1
    rng = np.random.default_rng(9)
    img = rng.standard_normal((h * w, cin), dtype=np.float32)
    filters = [O.f32_to_bf16((rng.standard_normal((cout, 9 * cin)) * 0.1).astype(np.float32)) for _ in range(2)]
    bias = rng.standard_normal(cout).astype(np.float32)
    want = [conv_float64(img, f, bias, h, w, 3, 1, 1, 1) for f in filters]
    x = O.f32_to_bf16(rng.standard_normal((rows, k)).astype(np.float32))
    weight = O.f32_to_bf16((rng.standard_normal((out, k)) * 0.05).astype(np.float32))
    want_layer = O.bf16_to_f32(x).astype(np.float64) @ O.bf16_to_f32(weight).astype(np.float64).T
    dimg, dbias, dx, dweight = dev.put(img), dev.put(bias), dev.put(x), dev.put(weight)
    f1, f2 = [dev.put(f) for f in filters]
    captured, eager, layer = dev.alloc(h * w * cout * 4), dev.alloc(h * w * cout * 4), dev.alloc(rows * out * 4)
    conv = lambda dst, f: lib.iris_dev_conv2d(dst, dimg, f, dbias, h, w, cin, cout, 3, 1, 1, 1)

    conv(eager, f2)
    dev.check()
    lib.iris_dev_sync()
    first = dev.get(eager, (h * w, cout), np.float32)
    run = g.capture(stream, lambda: conv(captured, f1))
    assert g.nodes == 1
    dev.check()
    lib.iris_dev_sync()
    other = _vp()
    assert g.rt.hipStreamCreate(C.byref(other)) == 0
    junk = np.full(h * w * cout, np.nan, np.float32)
    for replay in range(4):
        for p, n in ((captured, h * w * cout), (eager, h * w * cout), (layer, rows * out)):
            lib.iris_dev_upload(p, junk.ctypes.data_as(_vp), n * 4)
        for _ in range(8):
            assert g.rt.hipGraphLaunch(run, other) == 0
            conv(eager, f2)
            lib.iris_dev_linear_f32(layer, dx, dweight, rows, k, out)
        assert g.rt.hipStreamSynchronize(other) == 0
        lib.iris_dev_sync()
        dev.check()
        got = dev.get(eager, (h * w, cout), np.float32)
        assert np.array_equal(got, first)
        for v, e in ((dev.get(captured, (h * w, cout), np.float32), want[0]), (got, want[1])):
            np.testing.assert_allclose(v.reshape(e.shape), e, atol=2e-5 * np.sqrt(9 * cin))
        np.testing.assert_allclose(dev.get(layer, (rows, out), np.float32), want_layer, atol=2e-5 * np.sqrt(k) * 0.05)
    g.rt.hipGraphExecDestroy(run)
    g.rt.hipStreamDestroy(other)
    dev.free_all()
