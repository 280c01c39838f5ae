"""Row norms at both sides of the choices between a wave and a workgroup per row, with and without the row kept in
registers, against the CPU oracle (bf16 results: one unit in the last place, from the order of the f32 sums)."""
import numpy as np
import pytest

import oracle as O
from gpu_harness import Dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return Dev()


@pytest.mark.parametrize("rows,dim", [(2047, 64), (2048, 64), (2049, 128), (2051, 1024), (2048, 1028), (2049, 33), (2050, 1023), (3, 1024)])
def test_both_routes(dev, orc, rows, dim):
    compare(dev, orc, rows, dim)


# the last rows of a workgroup's and the first of a wave's, lengths that end inside and at the end of what a wave keeps, and as many
# long rows as LayerNorm deals out in waves again
@pytest.mark.parametrize("rows,dim", [(1280, 1024), (1281, 1024), (1283, 64), (1281, 1028), (1285, 1536), (1282, 1540), (1283, 2048), (1281, 2052),
                                      (32768, 2052), (32769, 1030)])
def test_edges_of_the_routes(dev, orc, rows, dim):
    compare(dev, orc, rows, dim)


def compare(dev, orc, rows, dim):
    rng = np.random.default_rng(rows + dim)
    x = (2 * rng.standard_normal((rows, dim)) + 0.7).astype(np.float32)
    p = [(0.3 * rng.standard_normal(dim) + at).astype(np.float32) for at in (0.0, 0.0, 1.0)]
    dx, (dsh, dsc, dw) = dev.put(x), (dev.put(v) for v in p)
    d1, d2, dres = dev.alloc(rows * dim * 2), dev.alloc(rows * dim * 2), dev.put(x)
    dev.lib.iris_dev_layer_norm_mod(d1, dx, dsh, dsc, rows, dim, 1e-6)
    dev.lib.iris_dev_rms_norm_mod(d2, dx, dw, dsc, rows, dim, 1e-5)
    dev.lib.iris_dev_rms_norm_residual(dres, dx, dw, dsc, rows, dim, 1e-6)
    dev.check()
    g1, g2, res = dev.get(d1, (rows, dim), np.uint16), dev.get(d2, (rows, dim), np.uint16), dev.get(dres, (rows, dim), np.float32)
    dev.free_all()
    for got, want in ((g1, orc.dev_layer_norm_mod(x, p[0], p[1], 1e-6)), (g2, orc.dev_rms_norm_mod(x, p[2], p[1], 1e-5))):
        want = want if want.dtype == np.uint16 else O.f32_to_bf16(want)
        # a value next to a rounding boundary may fall on the other side: 2^-8 of it
        a, b = O.bf16_to_f32(got), O.bf16_to_f32(want)
        np.testing.assert_allclose(a, b, rtol=2.0 ** -7, atol=1e-5)
        assert (got != want).mean() < 0.01
    np.testing.assert_allclose(res, orc.dev_rms_norm_residual(x, x, p[2], p[1], 1e-6), atol=5e-5)
