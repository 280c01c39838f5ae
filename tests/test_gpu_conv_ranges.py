"""3 x 3 convolutions whose last round of tiles is cut into ranges of input channels (k_conv_3x3 with a workspace), against the
definition in float64: one tile cut sixteen ways, ranges over two tiles, whole rounds in front, an XCD with more left over than the
others, ragged tiles, outputs that are not rows of 16 bytes, no bias."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from gpu_harness import Dev
from test_gpu_conv_direct import conv_float64

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import torch
    torch.cuda.init()
    return Dev()


@pytest.mark.parametrize("h,w,cin,cout,pb,pa,bias", [
    (16, 16, 1024, 128, 1, 1, True), (17, 15, 512, 130, 1, 1, True), (64, 69, 512, 256, 1, 1, False), (66, 70, 512, 200, 1, 0, True),
    (50, 47, 576, 513, 1, 1, True), (122, 131, 512, 512, 1, 1, True), (112, 592, 512, 128, 1, 1, True), (130, 270, 512, 130, 0, 1, False),
    (60, 30, 256, 128, 1, 1, True), (132, 141, 512, 512, 1, 1, True)])
def test_against_float64(dev, h, w, cin, cout, pb, pa, bias):
    oh, ow = h + pb + pa - 2, w + pb + pa - 2
    assert dev.lib.iris_hip_conv2d_cut(oh, ow, cin, cout) == 1
    rng = np.random.default_rng(h + w + cout)
    img = rng.standard_normal((h * w, cin), dtype=np.float32)
    wt = O.f32_to_bf16((rng.standard_normal((cout, 9 * cin)) * 0.1).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32) if bias else np.zeros(cout, np.float32)
    want = conv_float64(img, wt, b, h, w, 3, 1, pb, pa)
    out = dev.put(np.full(want.size + 64, 7.0, np.float32))
    args = dev.put(img), dev.put(wt), dev.put(b) if bias else None, h, w, cin, cout, 3, 1, pb, pa
    got = []
    for _ in range(2):
        dev.lib.iris_dev_conv2d(out, *args)
        dev.check()
        got.append(dev.get(out, (want.size + 64,), np.float32))
    dev.free_all()
    assert (got[0][want.size:] == 7.0).all() and np.array_equal(got[0], got[1])
    np.testing.assert_allclose(got[0][:want.size].reshape(want.shape), want, atol=2e-5 * np.sqrt(9 * cin))


@pytest.mark.parametrize("h,w", [(364, 360), (365, 360)])
def test_results_up_to_64_megabytes_are_written_through_and_larger_ones_are_not(dev, h, w):
    """Whole and ragged tiles of both: 128 channels of 131040 and of 131400 pixels."""
    cin, cout = 64, 128
    assert (h * w * cout * 4 <= 64 << 20) == (h == 364)
    rng = np.random.default_rng(h)
    img = rng.standard_normal((h * w, cin), dtype=np.float32)
    wt = O.f32_to_bf16((rng.standard_normal((cout, 9 * cin)) * 0.1).astype(np.float32))
    b = rng.standard_normal(cout).astype(np.float32)
    want = conv_float64(img, wt, b, h, w, 3, 1, 1, 1)
    out = dev.put(np.full(want.size + 64, 7.0, np.float32))
    dev.lib.iris_dev_conv2d(out, dev.put(img), dev.put(wt), dev.put(b), h, w, cin, cout, 3, 1, 1, 1)
    dev.check()
    got = dev.get(out, (want.size + 64,), np.float32)
    dev.free_all()
    assert (got[want.size:] == 7.0).all()
    np.testing.assert_allclose(got[:want.size].reshape(want.shape), want, atol=2e-5 * np.sqrt(9 * cin))
