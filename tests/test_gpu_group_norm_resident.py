"""Group norm as one launch (k_gn_resident), through its launcher so that every size takes it, against float64: workgroups with
no, one and all steps kept, in registers, in the LDS and beyond both, images that end inside a step, in place, and workgroups
that give up their share at once (patience 0: the last one to arrive does theirs) between ordinary calls on the same scratch."""
import ctypes as C

import numpy as np
import pytest

from gpu_harness import Dev

pytestmark = pytest.mark.gpu
WGS, REG, KEEP, BATCH = 256, 48, 66, 8                         # workgroups; steps of 2048 floats kept in registers, in all; read at a time
NOT_TAKEN = -2


@pytest.fixture(scope="module")
def dev():
    d = Dev()
    d.lib.iris_hip_group_norm_scratch_floats.restype = C.c_size_t
    d.stream = C.c_void_p(d.lib.iris_dev_stream())
    d.scratch = C.c_void_p(d.lib.iris_dev_alloc(4 * d.lib.iris_hip_group_norm_scratch_floats(64)))
    assert d.lib.iris_hip_group_norm_prepare_scratch(d.stream, d.scratch) == 0
    return d


def resident(dev, out, img, gamma, beta, hw, c, groups, silu, patience=1000000):
    ptrs = [C.c_void_p(p) for p in (out, img, gamma, beta)]
    return dev.lib.iris_hip_group_norm_resident(dev.stream, dev.scratch, *ptrs, hw, c, groups, C.c_float(1e-6), silu, C.c_uint(patience))


def data(hw, c):
    rng = np.random.default_rng(hw + c)
    x = rng.standard_normal((hw, c), dtype=np.float32) * 2 + 0.5 + 0.01 * np.arange(c, dtype=np.float32)
    return x, (1 + 0.1 * rng.standard_normal(c)).astype(np.float32), (0.1 * rng.standard_normal(c)).astype(np.float32)


def expected(x, gamma, beta, groups, silu):
    hw, c = x.shape
    y = x.astype(np.float64).reshape(hw, groups, c // groups)
    y -= y.mean(axis=(0, 2), keepdims=True)
    y /= np.sqrt((y ** 2).mean(axis=(0, 2), keepdims=True) + 1e-6)
    y = y.reshape(hw, c) * gamma + beta
    return y / (1 + np.exp(-y)) if silu else y


def compare(got, want):
    # f32: the mean, three products and a sum of values up to 6 are each off by half a unit in the last place, 2^-22 there, and
    # the statistics by a few 2^-24
    np.testing.assert_allclose(got, want, atol=6 * 2.0 ** -20)


def steps(n, c):
    """pixels of n steps"""
    return n * 2048 // c


# hw, c, groups, silu
CASES = [(1, 128, 32, 1), (15, 128, 32, 0), (17, 128, 32, 1), (steps(255, 512) + 1, 512, 32, 0), (steps(WGS, 128) - 3, 128, 32, 1),
         (steps(WGS * BATCH, 64) + 5, 64, 16, 0), (steps(WGS * BATCH + 1, 64), 64, 8, 1), (steps(WGS * 9, 256) + 3, 256, 64, 1),
         (steps(WGS * REG, 128), 128, 32, 0), (steps(WGS * REG + 7, 128) + 1, 128, 32, 1), (steps(WGS * (REG + 7), 256), 256, 32, 1),
         (steps(WGS * KEEP, 128), 128, 32, 1), (steps(WGS * KEEP, 128) + 1, 128, 32, 0), (steps(WGS * (KEEP + 1) + 40, 128) + 3, 128, 32, 1),
         (steps(WGS * (KEEP + BATCH) + 9, 512), 512, 32, 1), (steps(WGS * (KEEP + 3 * BATCH + 3), 128) + 7, 128, 32, 1)]


@pytest.mark.parametrize("hw,c,groups,silu", CASES)
def test_sizes(dev, hw, c, groups, silu):
    x, gamma, beta = data(hw, c)
    dx, dg, db = dev.put(x), dev.put(gamma), dev.put(beta)
    dout = dev.put(np.full((hw + 1, c), np.nan, np.float32))
    assert resident(dev, dout, dx, dg, db, hw, c, groups, silu) == 0
    assert resident(dev, dx, dx, dg, db, hw, c, groups, silu) == 0                           # in place
    got, same = dev.get(dout, (hw + 1, c), np.float32), dev.get(dx, (hw, c), np.float32)
    dev.free_all()
    compare(got[:hw], expected(x, gamma, beta, groups, silu))
    assert np.isnan(got[hw]).all()                                                           # nothing behind the image
    np.testing.assert_array_equal(got[:hw], same)


@pytest.mark.parametrize("hw,c", [(5, 128), (steps(WGS * 2 + 9, 128) + 3, 128), (steps(WGS * (KEEP + 1) + 5, 128) + 1, 128)])
def test_shares_that_are_given_up(dev, hw, c):
    """Counters and flags as an ordinary call leaves them: the same bits before, with and after impatient calls."""
    x, gamma, beta = data(hw, c)
    dx, dg, db, dout = dev.put(x), dev.put(gamma), dev.put(beta), dev.alloc(hw * c * 4)
    outs = []
    for patience in (1000000, 0, 0, 1000000, 0):
        dev.dev.lib.iris_dev_upload(dout, np.full((hw, c), np.nan, np.float32).ctypes.data_as(C.c_void_p), hw * c * 4)
        assert resident(dev, dout, dx, dg, db, hw, c, 32, 1, patience) == 0
        outs.append(dev.get(dout, (hw, c), np.float32))
    dev.free_all()
    compare(outs[0], expected(x, gamma, beta, 32, 1))
    for o in outs[1:]:
        np.testing.assert_array_equal(outs[0], o)


@pytest.mark.parametrize("hw,c", [(steps(WGS * 3, 128), 128), (steps(WGS + 40, 512) + 3, 512)])
def test_every_wave_stores_its_part_where_shares_are_given_up(dev, hw, c):
    """The last workgroup goes from its own share straight on to the others': its waves still have to know that it did not give
    up itself. Its share is another one in each call."""
    x, gamma, beta = data(hw, c)
    dx, dg, db, want = dev.put(x), dev.put(gamma), dev.put(beta), None
    douts = [dev.put(np.full((hw, c), np.nan, np.float32)) for _ in range(12)]
    for i, dout in enumerate(douts):
        assert resident(dev, dout, dx, dg, db, hw, c, 32, 1, 0 if i else 1000000) == 0
    for dout in douts:
        got = dev.get(dout, (hw, c), np.float32)
        want = got if want is None else want
        np.testing.assert_array_equal(got, want)
    dev.free_all()
    compare(want, expected(x, gamma, beta, 32, 1))


# words of 64 bits at the front of the scratch: arrivals of all launches with the number of those that gave up above bit 48, the
# last launch that all arrived in with that number in its low 16 bits; from byte 128 on the launch a workgroup gave up in
@pytest.mark.parametrize("launches,gone,flags", [(3, 0, 0), (3, 7, 3), (3, 7, 1), (1000, 65535, 1000), (1 << 32, 12, 1 << 32), ((1 << 32) - 1, 300, 5)])
def test_counters_that_calls_have_left_behind(dev, launches, gone, flags):
    """Shares given up in earlier launches, however many, are no business of this one: not normalised a second time in place."""
    hw, c = steps(WGS + 9, 128) + 3, 128
    x, gamma, beta = data(hw, c)
    dx, dg, db, dout = dev.put(x), dev.put(gamma), dev.put(beta), dev.alloc(hw * c * 4)
    words = np.zeros(16 + WGS, np.uint64)
    words[0], words[1], words[16:] = launches * WGS + (gone << 48), (launches << 16) + gone, flags
    dev.dev.lib.iris_dev_upload(dev.scratch, words.ctypes.data_as(C.c_void_p), words.nbytes)
    for patience in (1000000, 0):
        assert resident(dev, dout, dx, dg, db, hw, c, 32, 1, patience) == 0
        compare(dev.get(dout, (hw, c), np.float32), expected(x, gamma, beta, 32, 1))
    words = dev.get(dev.scratch, (16 + WGS,), np.uint64)
    assert words[0] % (1 << 48) == (launches + 2) * WGS and words[1] >> 16 == launches + 2 and words[1] % 65536 == words[0] >> 48
    assert resident(dev, dx, dx, dg, db, hw, c, 32, 1) == 0
    compare(dev.get(dx, (hw, c), np.float32), expected(x, gamma, beta, 32, 1))
    dev.free_all()
    assert dev.lib.iris_hip_group_norm_prepare_scratch(dev.stream, dev.scratch) == 0


@pytest.mark.parametrize("c,per_group", [(128, 4), (512, 16), (256, 32)])
@pytest.mark.parametrize("what", ["a hot pixel", "hot pixels", "a very hot pixel", "a hot row", "an offset", "a step"])
def test_values_far_from_the_rest(dev, c, per_group, what):
    """Where the sums of a thread start says nothing about the rest: images with pixels far off at the front of one workgroup's share
    or of all, with a large mean, with two levels."""
    hw = steps(WGS * 9, c)
    x, gamma, beta = data(hw, c)
    share = 2048 // c                                           # pixels from the front of a workgroup's share to that of the next
    if what == "a hot pixel": x[37 * share] += 600.0
    if what == "hot pixels": x[0:WGS * share:share] += 600.0
    if what == "a very hot pixel": x[37 * share] += 20000.0
    if what == "a hot row": x[:share] *= 30.0
    if what == "an offset": x += 1000.0
    if what == "a step": x[hw // 2:] += 200.0
    want = expected(x, gamma, beta, c // per_group, 0)
    dx, dg, db, dout = dev.put(x), dev.put(gamma), dev.put(beta), dev.alloc(hw * c * 4)
    assert resident(dev, dout, dx, dg, db, hw, c, c // per_group, 0) == 0
    got = dev.get(dout, (hw, c), np.float32)
    dev.free_all()
    # A thread adds 36 values and their squares about its first one, d of it away: M2 loses at most 36 d^2 x 2^-24, and d^2 is at
    # most what M2 of the group has anyway. Half of it in the reciprocal root, once more for the merging; the mean is a float.
    rel = 36 * 2.0 ** -24 + 2.0 ** -20
    spread = x.astype(np.float64).std()
    np.testing.assert_allclose(got, want, rtol=rel, atol=6 * 2.0 ** -20 + np.abs(x.mean(dtype=np.float64)) / spread * 1.5 * 2.0 ** -23)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("pixel", [0, 16, -1])
@pytest.mark.parametrize("steps_each", [0.125, 3])
def test_infinities_and_nan_spoil_their_group_only(dev, value, pixel, steps_each):
    """As the definition has it (x - mean is infinite or not a number, the variance is not a number), and the other form. The last
    pixel is all that its workgroup has of the last step, or of the image."""
    hw, c, groups = steps(int(WGS * steps_each), 128) + 1, 128, 32
    x, gamma, beta = data(hw, c)
    x[pixel, 13] = value                                        # group 3
    x[pixel, 40], x[pixel - 1, 41] = value, -value              # group 10
    dx, dg, db, dout = dev.put(x), dev.put(gamma), dev.put(beta), dev.alloc(hw * c * 4)
    assert resident(dev, dout, dx, dg, db, hw, c, groups, 0) == 0
    got = dev.get(dout, (hw, c), np.float32)
    dev.free_all()
    spoilt = np.isin(np.arange(c) // 4, (3, 10))
    assert np.isnan(got[:, spoilt]).all()
    x[:, spoilt] = 0.0
    compare(got[:, ~spoilt], expected(x, gamma, beta, groups, 0)[:, ~spoilt])


def test_what_it_does_not_take(dev):
    hw = 64
    p = dev.alloc(hw * 512 * 4 + 16)
    for c, groups, shift in ((96, 32, 0), (128, 4, 0), (512, 128, 0), (64, 32, 0), (128, 32, 4), (4096, 32, 0)):
        assert resident(dev, p + shift, p, p, p, hw, c, groups, 0) == NOT_TAKEN, (c, groups, shift)
    assert resident(dev, p, p, p, p, (1 << 28) // 32, 128, 32, 0) == NOT_TAKEN               # 4 GiB
    dev.free_all()


@pytest.mark.parametrize("hw", [16383, 16384, 20479, 20480])   # 10 MB: the first size that takes it, and the last that does not
def test_both_sides_of_the_line(dev, hw):
    x, gamma, beta = data(hw, 128)
    dx, dg, db, dout = dev.put(x), dev.put(gamma), dev.put(beta), dev.alloc(hw * 128 * 4)
    dev.lib.iris_dev_group_norm(dout, dx, dg, db, hw, 128, 32, 1e-6, 1)
    dev.check()
    got = dev.get(dout, (hw, 128), np.float32)
    dev.free_all()
    compare(got, expected(x, gamma, beta, 32, 1))


def test_replayed_from_a_graph(dev):
    from test_gpu_graph import Graphs
    hw, c, lib, g = 21000, 128, dev.lib, Graphs()
    x, gamma, beta = data(hw, c)
    dx, dg, db, dout, deager = dev.put(x), dev.put(gamma), dev.put(beta), dev.alloc(hw * c * 4), dev.alloc(hw * c * 4)
    norm = lambda out: lib.iris_dev_group_norm_noalloc(out, dx, dg, db, hw, c, 32, 1e-6, 1)
    norm(deager)
    want = dev.get(deager, (hw, c), np.float32)
    run = g.capture(dev.stream, lambda: norm(dout))
    for _ in range(4):
        lib.iris_dev_upload(dout, np.full((hw, c), np.nan, np.float32).ctypes.data_as(C.c_void_p), hw * c * 4)
        assert g.rt.hipGraphLaunch(run, dev.stream) == 0
        lib.iris_dev_sync()
        np.testing.assert_array_equal(dev.get(dout, (hw, c), np.float32), want)
        norm(deager)
        np.testing.assert_array_equal(dev.get(deager, (hw, c), np.float32), want)
    g.rt.hipGraphExecDestroy(run)
    dev.check()
    dev.free_all()
    compare(want, expected(x, gamma, beta, 32, 1))


def test_first_call_of_a_process_inside_a_relaxed_capture(tmp_path):
    """The counters are cleared by then: an eager call before the first replay, the replays and eager calls between them all give
    the same. A copy of the library, so that the call is its first."""
    import shutil
    import iris_c_amd
    from test_gpu_graph import Graphs
    lib = C.CDLL(shutil.copy(iris_c_amd.LIB_PATH, tmp_path / "first_call.so"))
    for name, (res, args) in iris_c_amd.ABI.items():
        getattr(lib, name).restype, getattr(lib, name).argtypes = res, args
    assert lib.iris_dev_init() == 1
    g, stream = Graphs(), C.c_void_p(lib.iris_dev_stream())
    hw, c = 40000, 128
    x, gamma, beta = data(hw, c)
    def put(a):
        p = lib.iris_dev_alloc(a.nbytes)
        lib.iris_dev_upload(p, a.ctypes.data_as(C.c_void_p), a.nbytes)
        return p
    dx, dg, db, captured, eager = put(x), put(gamma), put(beta), lib.iris_dev_alloc(x.nbytes), lib.iris_dev_alloc(x.nbytes)
    graph, run = C.c_void_p(), C.c_void_p()
    assert g.rt.hipStreamBeginCapture(stream, 2) == 0                                          # hipStreamCaptureModeRelaxed
    lib.iris_dev_group_norm(captured, dx, dg, db, hw, c, 32, 1e-6, 1)
    assert g.rt.hipStreamEndCapture(stream, C.byref(graph)) == 0 and graph
    assert lib.iris_dev_last_error() == 0
    assert g.rt.hipGraphInstantiate(C.byref(run), graph, None, None, 0) == 0
    g.rt.hipGraphDestroy(graph)
    got = np.empty_like(x)
    for _ in range(3):
        lib.iris_dev_group_norm(eager, dx, dg, db, hw, c, 32, 1e-6, 1)
        assert g.rt.hipGraphLaunch(run, stream) == 0
        lib.iris_dev_sync()
        for out in (eager, captured):
            lib.iris_dev_download(got.ctypes.data_as(C.c_void_p), out, got.nbytes)
            compare(got, expected(x, gamma, beta, 32, 1))
    g.rt.hipGraphExecDestroy(run)
    lib.iris_dev_cleanup()
