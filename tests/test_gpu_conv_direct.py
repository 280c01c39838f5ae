"""The convolutions that work straight on the f32 image (conv_gfx950.hip), at the sizes where their tiles and remainders
begin and end, against the CPU oracle (bf16-rounded operands, f32 sums: the bar is the rounding of the sum's order).
Larger images against the same sums in float64."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from gpu_harness import Dev, ptr_add

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return Dev()


def conv_case(dev, orc, h, w, cin, cout, k, stride, pb, pa, bias=True):
    rng = np.random.default_rng(h * 1000 + w + cout)
    img = rng.standard_normal((h * w, cin)).astype(np.float32)
    wt = O.f32_to_bf16((rng.standard_normal((cout, k * k * cin)) * 0.1).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32) if bias else np.zeros(cout, np.float32)
    want = orc.dev_conv2d(img, wt, b, h, w, k, stride, pb, pa)
    guard = 64                                               # floats behind the output that must stay as they are
    out = dev.put(np.full(want.size + guard, 7.0, np.float32))
    dev.lib.iris_dev_conv2d(out, dev.put(img), dev.put(wt), dev.put(b) if bias else None, h, w, cin, cout, k, stride, pb, pa)
    dev.check()
    got = dev.get(out, (want.size + guard,), np.float32)
    dev.free_all()
    assert (got[want.size:] == 7.0).all()
    np.testing.assert_allclose(got[:want.size].reshape(want.shape), want, atol=2e-5 * np.sqrt(k * k * cin))


@pytest.mark.parametrize("h,w,cin,cout,k,stride,pb,pa,bias", [
    (1, 1, 3, 128, 3, 1, 1, 1, True), (37, 29, 3, 128, 3, 1, 1, 1, True), (16, 5, 3, 130, 3, 1, 1, 1, False),
    (20, 21, 3, 260, 3, 2, 0, 1, True), (9, 9, 8, 64, 2, 1, 0, 0, True), (17, 3, 1, 12, 5, 1, 2, 2, True)])
def test_few_input_channels(dev, orc, h, w, cin, cout, k, stride, pb, pa, bias):
    conv_case(dev, orc, h, w, cin, cout, k, stride, pb, pa, bias)


@pytest.mark.parametrize("h,w,cout", [(247, 248, 512), (250, 250, 512), (245, 250, 516), (170, 181, 1024), (333, 65, 1500)])
def test_few_input_channels_wide_results_around_120_megabytes(dev, h, w, cout):
    """One store of a wave on its way from there on, written through in whole pieces of 128 channels or not"""
    rng = np.random.default_rng(cout)
    img = rng.standard_normal((h * w, 3)).astype(np.float32)
    wt = O.f32_to_bf16((rng.standard_normal((cout, 27)) * 0.1).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32)
    want = conv_float64(img, wt, b, h, w, 3, 1, 1, 1)
    out = dev.put(np.full(want.size + 64, 7.0, np.float32))
    dev.lib.iris_dev_conv2d(out, dev.put(img), dev.put(wt), dev.put(b), h, w, 3, cout, 3, 1, 1, 1)
    dev.check()
    got = dev.get(out, (want.size + 64,), np.float32)
    dev.free_all()
    assert (got[want.size:] == 7.0).all()
    np.testing.assert_allclose(got[:want.size].reshape(want.shape), want, atol=2e-5 * np.sqrt(27))


@pytest.mark.parametrize("h,w,cin,cout,k,stride,pb,pa,bias", [
    (1, 1, 128, 3, 3, 1, 1, 1, True), (16, 32, 128, 3, 3, 1, 1, 1, True), (17, 33, 128, 3, 3, 1, 1, 1, False),
    (40, 70, 32, 3, 3, 1, 1, 1, True), (15, 31, 64, 2, 3, 1, 0, 0, True), (33, 20, 64, 28, 1, 1, 0, 0, True),
    (21, 34, 128, 7, 2, 1, 0, 1, True)])
def test_few_output_channels(dev, orc, h, w, cin, cout, k, stride, pb, pa, bias):
    conv_case(dev, orc, h, w, cin, cout, k, stride, pb, pa, bias)


@pytest.mark.parametrize("h,w,cin,cout,k,pad", [(30000, 1, 128, 3, 1, 0), (1, 30000, 64, 3, 1, 0), (20000, 1, 32, 3, 3, 1), (3, 9000, 128, 3, 3, 1)])
def test_few_output_channels_of_images_thinner_than_a_tile(dev, orc, h, w, cin, cout, k, pad):
    conv_case(dev, orc, h, w, cin, cout, k, 1, pad, pad)


@pytest.mark.parametrize("h,w,cin,cout,pb,pa,bias", [
    (1, 1, 64, 128, 1, 1, True), (16, 16, 64, 128, 1, 1, True), (17, 15, 128, 128, 1, 1, False), (33, 47, 192, 256, 1, 1, True),
    (18, 19, 64, 130, 0, 0, True), (3, 34, 320, 37, 2, 1, True), (20, 5, 512, 512, 1, 1, True), (16, 33, 256, 3, 0, 1, False)])
def test_three_by_three(dev, orc, h, w, cin, cout, pb, pa, bias):
    """Tile edges (16 x 16 pixels, 128 channels), one to eight groups of 64 input channels, padding of other widths."""
    conv_case(dev, orc, h, w, cin, cout, 3, 1, pb, pa, bias)


@pytest.mark.parametrize("h,w,cin,cout,bias", [(1, 1, 128, 128, True), (8, 4, 128, 128, True), (257, 1, 256, 130, False), (33, 31, 512, 64, True),
                                               (300, 1, 512, 1536, True), (2000, 1, 512, 1536, True), (90, 91, 384, 256, True), (17, 16, 64, 320, True), (9, 9, 128, 258, True), (128, 128, 128, 3, False)])
def test_one_by_one(dev, orc, h, w, cin, cout, bias):
    """One block of 16 pixels and less, as many blocks as waves, one and two tiles of 128 channels, a ragged one; and what goes
    through the bf16 copy and a plain product with the bias in its epilogue or behind it."""
    conv_case(dev, orc, h, w, cin, cout, 1, 1, 0, 0, bias)


@pytest.mark.parametrize("h,w,cin,cout,pb,pa,bias", [
    (2, 2, 128, 128, 0, 1, True), (16, 32, 32, 128, 0, 1, True), (17, 33, 64, 128, 0, 0, False), (33, 32, 128, 130, 0, 1, True),
    (31, 67, 96, 256, 1, 1, True), (46, 44, 256, 256, 0, 1, True), (40, 41, 160, 260, 2, 0, False), (5, 200, 512, 129, 1, 0, True),
    (150, 340, 128, 256, 0, 1, True)])
def test_three_by_three_stride_two(dev, orc, h, w, cin, cout, pb, pa, bias):
    """Tile edges (8 x 16 output pixels, 128 channels), one to sixteen groups of 32 input channels (odd and even numbers of them),
    padding of other widths, nearly as many tiles as workgroups."""
    conv_case(dev, orc, h, w, cin, cout, 3, 2, pb, pa, bias)


@pytest.mark.parametrize("h,w,cin,cout,k,stride,pb,pa,shift", [
    (40, 50, 128, 128, 3, 1, 1, 1, 0), (40, 50, 128, 256, 3, 1, 1, 1, 4096), (33, 47, 256, 128, 1, 1, 0, 0, 0), (41, 37, 128, 256, 3, 2, 0, 1, 0),
    (60, 70, 128, 3, 3, 1, 1, 1, 0), (70, 60, 3, 128, 3, 1, 1, 1, 64), (90, 30, 64, 64, 3, 1, 1, 1, 0)])
def test_output_in_the_image_s_own_memory(dev, orc, h, w, cin, cout, k, stride, pb, pa, shift):
    """The result begins `shift` floats into the image: every route that such a call can take has read the image by then."""
    rng = np.random.default_rng(h + w + cout)
    img = rng.standard_normal((h * w, cin)).astype(np.float32)
    wt = O.f32_to_bf16((rng.standard_normal((cout, k * k * cin)) * 0.1).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32)
    want = orc.dev_conv2d(img, wt, b, h, w, k, stride, pb, pa)
    room = np.zeros(max(img.size, shift + want.size), np.float32)
    room[:img.size] = img.ravel()
    mem = dev.put(room)
    out = ptr_add(mem, 4 * shift)
    dev.lib.iris_dev_conv2d(out, mem, dev.put(wt), dev.put(b), h, w, cin, cout, k, stride, pb, pa)
    dev.check()
    got = dev.get(out, want.shape, np.float32)
    dev.free_all()
    np.testing.assert_allclose(got, want, atol=2e-5 * np.sqrt(k * k * cin))


@pytest.mark.parametrize("h,w,cin,cout,stride,pb,pa", [(1, 9000, 64, 384, 1, 1, 1), (8, 1100, 128, 640, 1, 1, 1), (9000, 1, 64, 40, 1, 1, 1),
                                                       (9000, 1, 128, 640, 2, 1, 1), (1, 2000, 128, 256, 1, 1, 1), (3, 700, 64, 256, 2, 0, 1)])
def test_three_by_three_of_images_thinner_than_a_tile(dev, orc, h, w, cin, cout, stride, pb, pa):
    """On both sides of the choice between the tiles and a copy of the image."""
    conv_case(dev, orc, h, w, cin, cout, 3, stride, pb, pa)


def conv_float64(img, wt, bias, h, w, k, stride, pb, pa):
    """The definition, tap by tap in float64 on the bf16-rounded operands, on the device."""
    import torch
    cin, cout = img.shape[1], wt.shape[0]
    oh, ow = (h + pb + pa - k) // stride + 1, (w + pb + pa - k) // stride + 1
    x = torch.zeros(h + pb + pa, w + pb + pa, cin, dtype=torch.float64, device="cuda")
    x[pb:pb + h, pb:pb + w] = torch.from_numpy(O.bf16_to_f32(O.f32_to_bf16(img)).reshape(h, w, cin)).cuda()
    taps = torch.from_numpy(O.bf16_to_f32(wt).reshape(cout, k, k, cin)).cuda().double()
    out = torch.from_numpy(bias).cuda().double().repeat(oh * ow, 1)
    for ky in range(k):
        for kx in range(k):
            pixels = x[ky:ky + stride * (oh - 1) + 1:stride, kx:kx + stride * (ow - 1) + 1:stride].reshape(oh * ow, cin)
            out += pixels @ taps[:, ky, kx].t().contiguous()
    return out.cpu().numpy()


FEW_IN, ONE_BY_ONE, THREE, THREE_HALF = 1, 3, 4, 5             # iris_hip_conv2d_plan


@pytest.mark.parametrize("kernel,turns,h,w,cin,cout,k,stride,pb,pa", [
    (FEW_IN, 2, 301, 290, 3, 128, 3, 1, 1, 1), (FEW_IN, 3, 500, 341, 3, 130, 3, 1, 1, 1), (FEW_IN, 2, 600, 580, 7, 260, 2, 2, 0, 0),
    (ONE_BY_ONE, 2, 70001, 1, 128, 100, 1, 1, 0, 0), (ONE_BY_ONE, 2, 211, 193, 256, 200, 1, 1, 0, 0), (ONE_BY_ONE, 3, 301, 233, 384, 256, 1, 1, 0, 0),
    (THREE, 2, 150, 250, 64, 260, 3, 1, 1, 1), (THREE, 2, 130, 270, 192, 130, 3, 1, 1, 1), (THREE, 4, 250, 270, 64, 384, 3, 1, 0, 1),
    (THREE_HALF, 2, 150, 340, 128, 260, 3, 2, 0, 1), (THREE_HALF, 2, 180, 360, 96, 130, 3, 2, 0, 1), (THREE_HALF, 2, 190, 350, 64, 256, 3, 2, 1, 1),
    (THREE_HALF, 3, 201, 399, 32, 400, 3, 2, 1, 0)])
def test_work_taken_in_several_turns(dev, kernel, turns, h, w, cin, cout, k, stride, pb, pa):
    """Waves and workgroups that go on to another piece, with what they keep between pieces: fetches ahead, another tile of
    channels, operand sets that change places (odd and even numbers of channel groups), ragged last pieces."""
    plan = (C.c_int * 2)()
    dev.lib.iris_hip_conv2d_plan(C.c_void_p(1 << 44), C.c_void_p(1 << 40), C.c_void_p(1 << 46), h, w, cin, cout, k, stride, pb, pa, plan)
    assert (plan[0], plan[1]) == (kernel, turns)
    rng = np.random.default_rng(h + w + cout)
    img = rng.standard_normal((h * w, cin), dtype=np.float32)
    wt = O.f32_to_bf16((rng.standard_normal((cout, k * k * cin)) * 0.1).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32)
    want = conv_float64(img, wt, b, h, w, k, stride, pb, pa)
    guard = 64
    out = dev.put(np.full(want.size + guard, 7.0, np.float32))
    dev.lib.iris_dev_conv2d(out, dev.put(img), dev.put(wt), dev.put(b), h, w, cin, cout, k, stride, pb, pa)
    dev.check()
    got = dev.get(out, (want.size + guard,), np.float32)
    dev.free_all()
    assert (got[want.size:] == 7.0).all()
    np.testing.assert_allclose(got[:want.size].reshape(want.shape), want, atol=2e-5 * np.sqrt(k * k * cin))


ZERO_BYTES = 256                                             # IRIS_CONV_ZERO_BYTES


# scratch: what it holds behind the page of zeros, in rows of the image, pixels or patches, as the route counts
@pytest.mark.parametrize("route,h,w,cin,cout,k,stride,pb,pa,scratch", [
    ("implicit", 37, 29, 64, 128, 5, 1, 2, 2, 9), ("implicit", 40, 33, 128, 260, 5, 2, 1, 3, 7), ("implicit", 30, 41, 192, 256, 2, 1, 0, 1, 2),
    ("implicit", 41, 30, 64, 384, 2, 2, 1, 0, 5), ("implicit", 50, 37, 64, 130, 3, 3, 1, 1, 8), ("implicit", 23, 21, 128, 320, 5, 1, 2, 2, 64),
    ("plain", 61, 13, 512, 320, 1, 1, 0, 0, 150), ("plain", 1000, 1, 576, 264, 1, 1, 0, 0, 333), ("plain", 20, 20, 512, 512, 1, 1, 0, 0, 400),
    ("gathered", 30, 31, 24, 64, 3, 1, 1, 1, 100), ("gathered", 31, 30, 5, 40, 3, 2, 0, 1, 77), ("gathered", 25, 26, 64, 60, 5, 1, 2, 2, 7),
    ("gathered", 19, 18, 72, 128, 2, 2, 0, 0, 1)])
def test_routes_that_copy_the_image_in_chunks_of_the_scratch(dev, route, h, w, cin, cout, k, stride, pb, pa, scratch):
    """The routes of gemm_conv_gfx950.hip with a scratch that holds only part of the copy (and once all of it): taps other than 3 x 3
    through the implicit product, chunks of output rows with their halo, of pixels, of gathered patches, ragged last ones."""
    row_bytes = {"implicit": w * cin, "plain": cin, "gathered": k * k * cin}[route] * 2
    scratch_bytes, guard = ZERO_BYTES + scratch * row_bytes, 256
    plan = (C.c_int * 2)()
    dev.lib.iris_hip_conv2d_plan(C.c_void_p(1 << 44), C.c_void_p(1 << 40), C.c_void_p(1 << 46), h, w, cin, cout, k, stride, pb, pa, plan)
    assert plan[0] == 0 and (route == "implicit") == (cin % 64 == 0 and cout >= 128 and k > 1)
    if route == "plain":
        dev.lib.iris_hip_linear_plan(min(h * w, scratch), cin, cout, 4, plan)
        assert plan[0] == 4
    rng = np.random.default_rng(h + w + cout)
    img = rng.standard_normal((h * w, cin)).astype(np.float32)
    wt = O.f32_to_bf16((rng.standard_normal((cout, k * k * cin)) * 0.1).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32)
    want = conv_float64(img, wt, b, h, w, k, stride, pb, pa)
    room = dev.put(np.full(scratch_bytes + guard, 0x5a, np.uint8))
    out = dev.put(np.full(want.size + 64, 7.0, np.float32))
    vp, ci = C.c_void_p, C.c_int
    stream = vp(dev.lib.iris_dev_stream())
    conv = dev.lib.iris_hip_conv2d
    conv.argtypes = [vp, vp, C.c_size_t, vp, vp, vp, vp] + [ci] * 8
    dev.lib.iris_hip_conv2d_prepare_scratch.argtypes = [vp, vp]
    assert dev.lib.iris_hip_conv2d_prepare_scratch(stream, room) == 0
    assert conv(stream, room, scratch_bytes, out, dev.put(img), dev.put(wt), dev.put(b), h, w, cin, cout, k, stride, pb, pa) == 0
    dev.check()
    got = dev.get(out, (want.size + 64,), np.float32)
    page = dev.get(room, (scratch_bytes + guard,), np.uint8)
    dev.free_all()
    assert (got[want.size:] == 7.0).all() and (page[scratch_bytes:] == 0x5a).all() and not page[:ZERO_BYTES].any()
    np.testing.assert_allclose(got[:want.size].reshape(want.shape), want, atol=2e-5 * np.sqrt(k * k * cin))


@pytest.mark.parametrize("h,w,cin,cout,k,stride,pb,pa", [
    (40, 33, 64, 128, 3, 1, 1, 1), (30, 31, 3, 128, 3, 1, 1, 1), (28, 26, 128, 3, 3, 1, 1, 1), (32, 24, 128, 128, 3, 2, 0, 1), (40, 70, 128, 128, 1, 1, 0, 0)])
def test_routes_that_copy_the_image_take_every_shape(dev, h, w, cin, cout, k, stride, pb, pa):
    """Also those that iris_dev_conv2d gives to kernels without a copy: asked once, by it, and not again on the way here."""
    plan = (C.c_int * 2)()
    dev.lib.iris_hip_conv2d_plan(C.c_void_p(1 << 44), C.c_void_p(1 << 40), C.c_void_p(1 << 46), h, w, cin, cout, k, stride, pb, pa, plan)
    assert plan[0] != 0
    rng = np.random.default_rng(h + w + cout)
    img = rng.standard_normal((h * w, cin)).astype(np.float32)
    wt = O.f32_to_bf16((rng.standard_normal((cout, k * k * cin)) * 0.1).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32)
    want = conv_float64(img, wt, b, h, w, k, stride, pb, pa)
    scratch_bytes = ZERO_BYTES + h * w * k * k * cin * 2
    room = dev.put(np.full(scratch_bytes, 0x5a, np.uint8))
    out = dev.put(np.full(want.size, 7.0, np.float32))
    vp, ci = C.c_void_p, C.c_int
    stream = vp(dev.lib.iris_dev_stream())
    conv = dev.lib.iris_hip_conv2d
    conv.argtypes = [vp, vp, C.c_size_t, vp, vp, vp, vp] + [ci] * 8
    dev.lib.iris_hip_conv2d_prepare_scratch.argtypes = [vp, vp]
    assert dev.lib.iris_hip_conv2d_prepare_scratch(stream, room) == 0
    assert conv(stream, room, scratch_bytes, out, dev.put(img), dev.put(wt), dev.put(b), h, w, cin, cout, k, stride, pb, pa) == 0
    dev.check()
    got = dev.get(out, want.shape, np.float32)
    page = dev.get(room, (scratch_bytes,), np.uint8)
    dev.free_all()
    assert not page[:ZERO_BYTES].any() and (page[ZERO_BYTES:ZERO_BYTES + 64] != 0x5a).any()
    np.testing.assert_allclose(got, want, atol=2e-5 * np.sqrt(k * k * cin))


def test_one_by_one_of_large_images(dev):
    """192 MB of pixels and a pixel less: the same bits, and those of the definition."""
    h, cin, cout = (192 << 20) // (384 * 4), 384, 100
    rng = np.random.default_rng(5)
    img = rng.standard_normal((h, cin), dtype=np.float32)
    wt = O.f32_to_bf16((rng.standard_normal((cout, cin)) * 0.1).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32)
    dimg, dw, db = dev.put(img), dev.put(wt), dev.put(b)
    got = []
    for n in (h, h - 1):
        out = dev.put(np.full((h + 1, cout), 7.0, np.float32))
        dev.lib.iris_dev_conv2d(out, dimg, dw, db, n, 1, cin, cout, 1, 1, 0, 0)
        dev.check()
        got.append(dev.get(out, (h + 1, cout), np.float32))
        assert (got[-1][n:] == 7.0).all()
    dev.free_all()
    np.testing.assert_array_equal(got[0][:h - 1], got[1][:h - 1])
    rows = np.unique(np.r_[0:40, h - 40:h, rng.integers(0, h, 400)])
    want = O.bf16_to_f32(O.f32_to_bf16(img[rows])).astype(np.float64) @ O.bf16_to_f32(wt).astype(np.float64).T + b
    np.testing.assert_allclose(got[0][rows], want, atol=2e-5 * np.sqrt(cin))
