"""iris_dev_upsample2x at channel counts on both sides of the 16-byte stores, odd sizes and unaligned images: exact copies."""
import numpy as np
import pytest

from gpu_harness import Dev, ptr_add

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return Dev()


@pytest.mark.parametrize("shift", [0, 1], ids=["aligned", "unaligned"])
@pytest.mark.parametrize("h,w,c", [(1, 1, 4), (3, 5, 1), (7, 3, 3), (5, 9, 4), (33, 17, 8), (2, 65, 12), (1, 7, 130), (9, 1, 64)])
def test_every_output_is_its_input_pixel(dev, orc, h, w, c, shift):
    img = np.random.default_rng(h + w + c).standard_normal((h * w, c)).astype(np.float32)
    n, guard = 4 * img.size, 64
    src = dev.put(np.concatenate([np.zeros(shift, np.float32), img.ravel()]))
    dst = dev.put(np.full(shift + n + guard, 7.0, np.float32))
    dev.lib.iris_dev_upsample2x(ptr_add(dst, 4 * shift), ptr_add(src, 4 * shift), h, w, c)
    dev.check()
    got = dev.get(dst, (shift + n + guard,), np.float32)
    dev.free_all()
    assert (got[:shift] == 7.0).all() and (got[shift + n:] == 7.0).all()
    np.testing.assert_array_equal(got[shift:shift + n].reshape(4 * h * w, c), orc.dev_upsample2x(img, h, w))
