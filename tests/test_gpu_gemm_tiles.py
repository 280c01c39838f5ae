"""k_gemm_tiles (gemm_tiles_gfx950.hip): every tile and K ranges at their edges, against a float64 product of the same bf16
operands. The bar is that of the other linear kernels: f32 accumulation noise for f32 outputs, half a bf16 ulp more for bf16."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from gpu_harness import Dev

pytestmark = pytest.mark.gpu
WIDE_ODD = [(513, 576, 17408), (600, 704, 20488), (2100, 1088, 6152), (512, 576, 19456)]
TILES = [(128, 128), (128, 192), (128, 256), (64, 256), (160, 192), (160, 256)]


@pytest.fixture(scope="module")
def dev():
    return Dev()


def operands(rows, k, out):
    rng = np.random.default_rng(rows * 7 + k + out)
    x = O.f32_to_bf16(rng.standard_normal((rows, k)).astype(np.float32))
    W = O.f32_to_bf16((rng.standard_normal((out, k)) * 0.05).astype(np.float32))
    return x, W, O.bf16_to_f32(x).astype(np.float64) @ O.bf16_to_f32(W).astype(np.float64).T


def check(got, want, k, bf16):
    scale = np.sqrt(k) * 0.05
    if bf16:
        assert np.all(np.abs(O.bf16_to_f32(got) - want) <= np.abs(want) * 2.0 ** -8 * 1.01 + scale * 2e-5)
    else:
        assert np.abs(got - want).max() <= scale * 2e-5


# rows and columns beyond whole tiles (the last tile holds 1 .. all but one row), k tiles: fewer than, as many as and one more
# than the ring holds, odd and even numbers of them, ranges of unequal length
@pytest.mark.parametrize("shape", range(len(TILES)))
@pytest.mark.parametrize("more_rows,more_cols,k,splits", [(0, 0, 64, 1), (1, 8, 128, 1), (-1, -8, 192, 1), (0, 72, 256, 1), (33, 0, 320, 1),
                                                          (-63, 8, 704, 3), (0, 0, 640, 2), (1, 8, 832, 6)])
@pytest.mark.parametrize("bf16", [False, True])
def test_every_tile(dev, shape, more_rows, more_cols, k, splits, bf16):
    rows, out = TILES[shape][0] + more_rows, TILES[shape][1] + more_cols
    x, W, want = operands(rows, k, out)
    lib = dev.lib
    lib.iris_hip_gemm_tiles.restype = C.c_int
    lib.iris_hip_gemm_tiles.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_void_p, C.c_void_p] + [C.c_int] * 3 + [C.c_void_p] + [C.c_int] * 2 + [C.c_void_p]
    guard = 512
    fill = np.full(rows * out + guard, 7, np.uint16 if bf16 else np.float32)
    dy, part = dev.put(fill), dev.alloc(splits * rows * out * 4)
    assert lib.iris_hip_gemm_tiles(lib.iris_dev_stream(), dy, 2 if bf16 else 4, dev.put(x), dev.put(W), rows, out, k, None, shape, splits, part) == 0
    dev.check()
    got = dev.get(dy, fill.shape, fill.dtype)
    dev.free_all()
    assert (got[rows * out:] == 7).all()
    check(got[:rows * out].reshape(rows, out), want, k, bf16)


def one_layer(dev, shape, rows, k, out, splits, bf16):
    x, W, want = operands(rows, k, out)
    lib = dev.lib
    lib.iris_hip_gemm_tiles.restype = C.c_int
    lib.iris_hip_gemm_tiles.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_void_p, C.c_void_p] + [C.c_int] * 3 + [C.c_void_p] + [C.c_int] * 2 + [C.c_void_p]
    fill = np.full(rows * out + 512, 7, np.uint16 if bf16 else np.float32)
    dy, part = dev.put(fill), dev.alloc(splits * rows * out * 4)
    assert lib.iris_hip_gemm_tiles(lib.iris_dev_stream(), dy, 2 if bf16 else 4, dev.put(x), dev.put(W), rows, out, k, None, shape, splits, part) == 0
    dev.check()
    got = dev.get(dy, fill.shape, fill.dtype)
    dev.free_all()
    assert (got[rows * out:] == 7).all()
    check(got[:rows * out].reshape(rows, out), want, k, bf16)


# the tile of 160 x 224 at the same edges
@pytest.mark.parametrize("more_rows,more_cols,k,splits", [(0, 0, 64, 1), (1, 8, 128, 1), (-1, -8, 192, 1), (0, 72, 256, 1), (33, 0, 320, 1),
                                                          (-63, 8, 704, 3), (0, 0, 640, 2), (1, 8, 832, 6)])
@pytest.mark.parametrize("bf16", [False, True])
def test_tile_of_224_columns(dev, more_rows, more_cols, k, splits, bf16):
    one_layer(dev, 6, 160 + more_rows, k, 224 + more_cols, splits, bf16)


# the tile of 128 x 96 at the same edges, and whole and partial groups of four k tiles (weights of at most 1 MB: in one order)
@pytest.mark.parametrize("rows,k,out,splits", [(128, 64, 96, 1), (129, 128, 104, 1), (127, 192, 88, 1), (128, 256, 168, 1), (161, 320, 96, 1), (65, 704, 104, 3),
                                               (128, 640, 96, 2), (129, 832, 104, 6), (637, 192, 472, 1), (637, 448, 472, 1), (637, 1216, 472, 4)])
@pytest.mark.parametrize("bf16", [False, True])
def test_tile_of_96_columns(dev, rows, k, out, splits, bf16):
    one_layer(dev, 7, rows, k, out, splits, bf16)


# five by five tiles: no whole group of four k tiles, one, several, and some left over; ranges of K with all of these. The weights are
# at most 3 MB, so all workgroups take them in one order: the different orders are the next test's
@pytest.mark.parametrize("shape", range(7))
@pytest.mark.parametrize("k_tiles,splits", [(3, 1), (4, 1), (7, 1), (13, 1), (16, 1), (19, 4)])
def test_orders_of_the_k_tiles(dev, shape, k_tiles, splits):
    tm, tn = (TILES + [(160, 224)])[shape]
    one_layer(dev, shape, 5 * tm - 3, 64 * k_tiles, 5 * tn - 8, splits, k_tiles % 2 == 0)


# the same with weights of more than the 4 MB of an L2, the only ones that are taken in different orders; just below them
@pytest.mark.parametrize("shape", range(8))
@pytest.mark.parametrize("more,splits", [(-2, 1), (1, 1), (2, 1), (3, 1), (4, 5)])
def test_orders_of_the_k_tiles_of_large_weights(dev, shape, more, splits):
    tm, tn = (TILES + [(160, 224), (128, 96)])[shape]
    out = 5 * tn - 8
    k = ((1 << 21) // out // 256 * 4 + more) * 64            # whole groups of four k tiles up to 4 MB, and `more` k tiles
    k += 256 * (more > 0 and k * out <= 1 << 21)
    assert (k * out > 1 << 21) == (more > 0)
    one_layer(dev, shape, 5 * tm - 3, k, out, splits, more % 2 == 0)


# up to eight partial sums are requested at once, more one after the other; the last workgroup is not full
@pytest.mark.parametrize("splits", [2, 3, 4, 5, 6, 7, 8, 9, 13])
@pytest.mark.parametrize("bf16", [False, True])
def test_numbers_of_partial_sums(dev, splits, bf16):
    one_layer(dev, 0, 131, 64 * 13, 136, splits, bf16)


@pytest.mark.parametrize("rows,k,out", [(1, 512, 128), (77, 2048, 1544), (130, 1536, 136), (300, 4096, 640), (500, 1024, 3072)])
@pytest.mark.parametrize("bf16", [False, True])
def test_linear_layers_that_take_it(dev, rows, k, out, bf16):
    plan = (C.c_int * 2)()
    dev.lib.iris_hip_linear_plan(rows, k, out, 2 if bf16 else 4, plan)
    assert plan[0] == 4
    x, W, want = operands(rows, k, out)
    dy = dev.alloc(rows * out * (2 if bf16 else 4))
    fn = dev.lib.iris_dev_linear_bf16 if bf16 else dev.lib.iris_dev_linear_f32
    for _ in range(2):                                       # the second call finds the first one's partial sums in the workspace
        fn(dy, dev.put(x), dev.put(W), rows, k, out)
    dev.check()
    got = dev.get(dy, (rows, out), np.uint16 if bf16 else np.float32)
    dev.free_all()
    check(got, want, k, bf16)


def test_without_a_workspace_k_stays_whole(dev):
    rows, k, out = 300, 4096, 640
    x, W, want = operands(rows, k, out)
    lib = dev.lib
    lib.iris_hip_linear_f32.restype = C.c_int
    lib.iris_hip_linear_f32.argtypes = [C.c_void_p] * 5 + [C.c_int] * 3
    dy = dev.alloc(rows * out * 4)
    assert lib.iris_hip_linear_f32(lib.iris_dev_stream(), None, dy, dev.put(x), dev.put(W), rows, k, out) == 0
    dev.check()
    got = dev.get(dy, (rows, out), np.float32)
    dev.free_all()
    check(got, want, k, False)


@pytest.mark.parametrize("rows,k,out", [(512, 128, 19456), (449, 384, 18448), (257, 256, 20480)])
@pytest.mark.parametrize("bf16", [False, True])
def test_wide_tiles_of_160_columns(dev, rows, k, out, bf16):
    """k_gemm_wide's narrowest tile: two to six k tiles, a last tile of one row, of 48 and of 96 columns."""
    plan = (C.c_int * 2)()
    dev.lib.iris_hip_linear_plan(rows, k, out, 2 if bf16 else 4, plan)
    assert list(plan) == [3, 160]
    x, W, want = operands(rows, k, out)
    guard = 512
    fill = np.full(rows * out + guard, 7, np.uint16 if bf16 else np.float32)
    dy = dev.put(fill)
    (dev.lib.iris_dev_linear_bf16 if bf16 else dev.lib.iris_dev_linear_f32)(dy, dev.put(x), dev.put(W), rows, k, out)
    dev.check()
    got = dev.get(dy, fill.shape, fill.dtype)
    dev.free_all()
    assert (got[rows * out:] == 7).all()
    check(got[:rows * out].reshape(rows, out), want, k, bf16)


@pytest.mark.parametrize("rows,k,out", WIDE_ODD)
@pytest.mark.parametrize("bf16", [False, True])
def test_wide_tiles_of_an_odd_number_of_k_tiles(dev, rows, k, out, bf16):
    plan = (C.c_int * 2)()
    dev.lib.iris_hip_linear_plan(rows, k, out, 2 if bf16 else 4, plan)
    assert plan[0] == 3
    x, W, want = operands(rows, k, out)
    dy = dev.alloc(rows * out * (2 if bf16 else 4))
    (dev.lib.iris_dev_linear_bf16 if bf16 else dev.lib.iris_dev_linear_f32)(dy, dev.put(x), dev.put(W), rows, k, out)
    dev.check()
    got = dev.get(dy, (rows, out), np.uint16 if bf16 else np.float32)
    dev.free_all()
    check(got, want, k, bf16)


@pytest.mark.parametrize("rows,out", [(131400, 264), (264, 131400)])
def test_wide_tiles_of_operands_beyond_four_gibibytes(dev, rows, out):
    """x or W of 4.3 GB: rows on both sides of the byte that 32 bits no longer count, against float64 products on the device."""
    import torch
    k = 16384
    plan = (C.c_int * 2)()
    dev.lib.iris_hip_linear_plan(rows, k, out, 4, plan)
    assert plan[0] == 3 and max(rows, out) * k * 2 > 1 << 32
    torch.manual_seed(4)
    x, W = torch.randn(rows, k, dtype=torch.bfloat16, device="cuda"), torch.randn(out, k, dtype=torch.bfloat16, device="cuda") * 0.05
    y = torch.empty(rows, out, device="cuda")
    torch.cuda.synchronize()
    dev.lib.iris_dev_linear_f32(y.data_ptr(), x.data_ptr(), W.data_ptr(), rows, k, out)
    dev.lib.iris_dev_sync()
    dev.check()
    pick = lambda n: torch.tensor(sorted({i % n for i in (0, 1, 255, 256, 131070, 131071, 131072, 131073, -257, -1)}), device="cuda")
    m, n = pick(rows), pick(out)
    want = x[m].double() @ W[n].double().t().contiguous()
    assert float((y[m][:, n].double() - want).abs().max()) <= np.sqrt(k) * 0.05 * 2e-5
    del x, W, y
    torch.cuda.empty_cache()


def test_projection_with_norm_takes_the_same_kernel(dev):
    """The projection that normalises its own columns, at a size whose plain layer takes these tiles: the bits of the two calls."""
    rows, k, heads = 320, 1024, 6
    out = 3 * heads * 128
    rng = np.random.default_rng(3)
    x, W, _ = operands(rows, k, out)
    w = [dev.put((1 + 0.05 * rng.standard_normal(128)).astype(np.float32)) for _ in range(2)]
    ang = rng.uniform(-3, 3, (rows, 64)).astype(np.float32)
    cos, sin, dx, dW = dev.put(np.cos(ang)), dev.put(np.sin(ang)), dev.put(x), dev.put(W)
    one, two = dev.alloc(rows * out * 2), dev.alloc(rows * out * 2)
    dev.lib.iris_dev_linear_bf16_qknorm(one, dx, dW, rows, k, out, heads, heads, 128, w[0], w[1], cos, sin, 1e-6, 0)
    assert dev.dev.last_kernel() == "linear_mfma_qknorm"
    dev.lib.iris_dev_linear_bf16(two, dx, dW, rows, k, out)
    dev.lib.iris_dev_head_norm_rope_qk(two, C.c_void_p(two + 2 * heads * 128), out, w[0], w[1], cos, sin, rows, heads, heads, 128, 1e-6, 0)
    dev.check()
    a, b = dev.get(one, (rows, out), np.uint16), dev.get(two, (rows, out), np.uint16)
    dev.free_all()
    assert np.array_equal(a, b)
