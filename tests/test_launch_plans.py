"""The launchers' choices are host arithmetic: which workgroup shape an attention problem gets, and for the two-size
grid how many workgroups of 256 and of 192 queries per head (iris_hip_fa_hd128_plan); which GEMM kernel and tile width
a linear layer gets (iris_hip_linear_plan). Runs without a GPU: the library loads, nothing is launched."""
import ctypes as C

import pytest

import iris_c_amd


@pytest.fixture(scope="module")
def plan():
    lib = C.CDLL(iris_c_amd.LIB_PATH)
    lib.iris_hip_fa_hd128_plan.argtypes = [C.c_int] * 4 + [C.POINTER(C.c_int)]
    lib.iris_hip_fa_hd128_plan.restype = None

    def call(seq_q, seq_k, heads, causal=0):
        out = (C.c_int * 5)()
        lib.iris_hip_fa_hd128_plan(seq_q, seq_k, heads, causal, out)
        return dict(kind=out[0], waves=out[1], nb=out[2], full=out[3], tails=out[4])
    return call


def test_benchmark_configurations(plan):
    assert plan(320, 320, 24) == dict(kind=0, waves=2, nb=1, full=0, tails=0)            # C1: 480 waves of 16 queries
    assert plan(512, 512, 32, 1) == dict(kind=0, waves=4, nb=1, full=0, tails=0)         # C4: 1024 such waves
    assert plan(4608, 4608, 24) == dict(kind=1, waves=8, nb=2, full=10, tails=11)        # C2: 432 x 256 queries = 1.69 rounds
    assert plan(4352, 4352, 30) == dict(kind=0, waves=8, nb=2, full=0, tails=0)          # C3: 510 workgroups, two full rounds
    p = plan(12800, 12800, 24)                                                            # C5: 4.69 rounds
    assert p["kind"] == 1 and 256 * p["full"] + 192 * p["tails"] >= 12800 and 24 * p["full"] <= 4 * 256


def test_short_sequences_split_the_keys_when_workgroups_are_few(plan):
    assert plan(512, 512, 1)["kind"] == 2 and plan(512, 512, 1)["waves"] == 4             # 8 key tiles: four waves
    assert plan(32, 448, 8)["kind"] == 2                                                  # 7 tiles: two turns of four waves + merge
    assert plan(128, 200, 4)["kind"] == 0                                                 # 4 tiles: the chain is shorter than a merge
    assert plan(64, 64, 8)["kind"] == 0                                                   # one key tile: nothing to split
    assert plan(512, 512, 32)["kind"] == 0                                                # 512 (head, 32-query block) pairs > 256 CUs


@pytest.mark.parametrize("heads", [8, 16, 20, 24, 30, 32, 40, 48])
def test_two_size_grids_cover_every_query_and_never_lose_to_one_size(plan, heads):
    kinds = set()
    for seq in list(range(2048 * 16 // heads + 64, 9000, 331)) + list(range(2048 * 16 // heads + 40, 9000, 197)):
        p = plan(seq, seq, heads)
        assert p["waves"] in (4, 8) and p["nb"] == 2, (seq, p)
        if p["kind"] == 1:
            assert p["full"] >= 0 and p["tails"] >= 0 and 256 * p["full"] + 192 * p["tails"] >= seq, (seq, p)
            assert 256 * p["full"] <= seq and 192 * (p["tails"] - 1) < seq - 256 * p["full"], (seq, p)     # no empty workgroup
            # priced per shader engine (8 CUs, a 192-query workgroup at 0.78): never above the rounds of the 8-wave kernel
            full_x, tail_x = -(-p["full"] * heads // 8), -(-p["tails"] * heads // 8)
            rounds_one_size = -(-(-(-seq // 256) * heads) // 256)
            per_engine = -(-(full_x + tail_x) // 4)
            assert per_engine <= 8 * (rounds_one_size + 1), (seq, p)
        if p["kind"] == 3:
            assert p["full"] >= 0 and 256 * p["full"] <= seq, (seq, p)
            assert 64 * (p["tails"] - 1) < seq - 256 * p["full"] <= 64 * p["tails"], (seq, p)
            # a 64-query workgroup at 0.33 and two key tiles of a 256-query one: dealt evenly they take 5 % less than whole rounds of one size
            tail = 33 + 200 // -(-seq // 64)
            assert heads * (100 * p["full"] + tail * p["tails"]) <= 256 * 95 * -(-(-(-seq // 256) * heads) // 256), (seq, p)
        kinds.add(p["kind"])
        assert plan(seq, seq, heads, 1)["kind"] == 0                                      # causal calls keep one size
    assert {1, 3} <= kinds


def test_a_few_workgroups_over_a_round_become_small_ones(plan):
    """256-query workgroups and 64-query ones behind them: every query in one of them, no empty workgroup"""
    for heads, seq in ((24, 2704), (24, 3264), (30, 2400), (32, 2064), (32, 2560), (16, 4112), (8, 8208), (48, 1296), (64, 1100), (30, 4864)):
        p = plan(seq, seq, heads)
        assert p["kind"] == 3 and p["waves"] == 8 and 256 * p["full"] <= seq, (heads, seq, p)
        assert 64 * (p["tails"] - 1) < seq - 256 * p["full"] <= 64 * p["tails"], (heads, seq, p)
    for heads, seq in ((24, 2627), (24, 3584), (24, 4608), (30, 5440), (24, 9536), (32, 4352), (24, 12800)):
        assert plan(seq, seq, heads)["kind"] in (0, 1), (heads, seq)


def test_small_workgroups_behind_a_key_mask_only_in_two_rounds(masked_kind):
    for heads, seq in ((24, 2816), (30, 2400), (32, 2304), (40, 1700)):
        assert masked_kind(heads, seq, 0) == masked_kind(heads, seq, 1) == 3
    for heads, seq in ((40, 3136), (30, 4816), (48, 2600)):
        assert masked_kind(heads, seq, 0) == 3 and masked_kind(heads, seq, 1) != 3


@pytest.fixture(scope="module")
def masked_kind():
    lib = C.CDLL(iris_c_amd.LIB_PATH)
    lib.iris_hip_fa_hd128_route.argtypes = [C.c_int] * 5 + [C.POINTER(C.c_int)]
    lib.iris_hip_fa_hd128_route.restype = None

    def call(heads, seq, masked):
        out = (C.c_int * 6)()
        lib.iris_hip_fa_hd128_route(seq, seq, heads, 0, masked, out)
        return out[0]
    return call


def test_exact_rounds_keep_one_size(plan):
    for heads, seq in ((16, 4096), (32, 2048), (8, 8192), (32, 4096), (30, 4352)):
        assert plan(seq, seq, heads)["kind"] == 0, (heads, seq)


@pytest.fixture(scope="module")
def parts():
    lib = C.CDLL(iris_c_amd.LIB_PATH)
    lib.iris_hip_fa_hd128_route.argtypes = [C.c_int] * 5 + [C.POINTER(C.c_int)]
    lib.iris_hip_fa_hd128_route.restype = None

    def call(seq_q, seq_k, heads, causal=0, masked=0):
        """waves with queries of their own, and that share theirs, of the kernel with one size of workgroups"""
        out = (C.c_int * 6)()
        lib.iris_hip_fa_hd128_route(seq_q, seq_k, heads, causal, masked, out)
        return (out[1], out[5]) if out[0] == 0 else None
    return call


def test_two_waves_share_their_queries_where_that_halves_a_chain_and_every_workgroup_has_a_cu(parts):
    assert parts(192, 192, 24) == (2, 1) and parts(193, 193, 24) == (2, 2)               # three key tiles; four
    assert parts(320, 320, 24) == (2, 2) and parts(321, 321, 24) == (4, 2)               # 240 workgroups of 32 queries; 264: 144 of 64
    assert parts(640, 640, 24) == (4, 2) and parts(641, 641, 24) == (4, 1)               # 240 workgroups of 64 queries; 264
    assert parts(320, 320, 24, 1) == (2, 2) and parts(512, 512, 32, 1) == (4, 2)
    assert parts(4352, 4352, 30) == (8, 1) and parts(64, 64, 24) == (1, 1)


def test_two_waves_share_their_queries_only_where_the_number_of_tiles_is_known_and_enough(parts):
    for heads, seq in ((24, 200), (24, 320), (24, 512), (30, 350), (32, 512), (40, 320)):
        assert parts(seq, seq, heads)[1] == 2
        for causal in (0, 1):
            assert parts(seq, seq, heads, causal, 1)[1] == 1                             # the walk ends at the last valid key
    for heads in (40, 48, 64):                                                           # 64 queries a workgroup, three tiles and a short fourth
        assert [parts(seq, seq, heads, 1)[1] for seq in (193, 208, 224, 225, 256)] == [1, 1, 1, 2, 2]
        assert parts(193, 193, heads)[1] == 2
    assert parts(193, 193, 24, 1) == (2, 2)


def test_causal_walks_behind_a_key_mask_get_smaller_workgroups_over_a_round(parts):
    """the walks may be short: with eight waves of 16 queries a workgroup they start late"""
    for heads, seq in ((32, 1025), (32, 1100), (32, 1152), (24, 1380), (24, 1536), (20, 1664)):
        assert parts(seq, seq, heads, 1, 1) == (4, 1) and parts(seq, seq, heads, 1, 0) == (8, 1)
    for heads, seq in ((32, 1024), (24, 1280), (16, 2048), (16, 2049), (16, 2300), (8, 4128)):   # one round; long walks
        assert parts(seq, seq, heads, 1, 1) == (8, 1)


# ------------------------------------------------------------------ the linear layers' kernel choice
@pytest.fixture(scope="module")
def linear_plan():
    lib = C.CDLL(iris_c_amd.LIB_PATH)
    lib.iris_hip_linear_plan.argtypes = [C.c_int] * 4 + [C.POINTER(C.c_int)]
    lib.iris_hip_linear_plan.restype = None

    def call(rows, k, out, out_bytes=2):
        p = (C.c_int * 2)()
        lib.iris_hip_linear_plan(rows, k, out, out_bytes, p)
        return p[0], p[1]
    return call


def test_linear_layers_of_the_models_take_the_wide_kernel_in_the_width_that_fills_the_rounds(linear_plan):
    assert linear_plan(4608, 3072, 9216) == (3, 224)        # 756 tiles = 2.95 rounds of 256 CUs (648 of 256 columns: 2.53)
    assert linear_plan(4608, 3072, 3072) == (3, 224)        # 252 tiles: one round (216 of 256 columns: also one, but wider)
    assert linear_plan(4608, 3072, 27648) == (3, 256)       # 1944 tiles = 7.6 rounds; narrower tiles need 9 or 11
    assert linear_plan(4608, 3072, 18432)[1] in (224, 192)  # 1296 tiles of 256 columns are 5.06 rounds
    for rows, k, out in ((300, 128, 258), (257, 64, 257), (512, 192, 256)):
        assert linear_plan(rows, k, out)[0] == 2             # rows of 2 bytes not 16-byte aligned, or three k tiles
    assert linear_plan(700, 256, 1000) == (3, 256) or linear_plan(700, 256, 1000)[0] == 3
    assert linear_plan(64, 128, 64)[0] == 1 and linear_plan(37, 27, 19)[0] == 0
    assert linear_plan(512, 256, 258, 4)[0] == 2             # f32 rows of 258 columns cannot take 16-byte stores


def test_long_products_of_an_odd_number_of_k_tiles_take_the_wide_kernel_too(linear_plan):
    for k in (576, 704, 1088, 2624, 3136):
        for out in (3072, 9216):
            assert linear_plan(4608, k, out)[0] == linear_plan(9000, k, out, 4)[0] == 3, (k, out)
    for k in (64, 192, 320, 448):
        assert linear_plan(4608, k, 9216)[0] == 2                  # the other kernel is as fast


def test_operands_of_four_gibibytes_and_more_take_the_wide_kernel(linear_plan):
    assert linear_plan(140000, 16384, 512)[0] == linear_plan(512, 16384, 140000, 4)[0] == 3
    assert linear_plan(300000, 8192, 300000)[0] == 3


def test_long_grids_of_large_products_take_the_wide_kernel(linear_plan):
    for rows, k, out, size in ((12800, 12288, 3072, 4), (12304, 9216, 3072, 4), (9280, 12288, 4096, 4), (9000, 16384, 4096, 4), (7176, 16384, 4096, 4),
                               (6100, 16384, 4096, 4), (6000, 12288, 4096, 4), (3640, 4096, 36864, 2), (4630, 3072, 18432, 2), (9500, 9728, 2560, 4)):
        assert linear_plan(rows, k, out, size)[0] == 3, (rows, k, out)
    for rows, k, out, size in ((5760, 9216, 3072, 4), (4160, 12288, 4096, 4), (12600, 4096, 4096, 4), (3640, 3072, 27648, 2)):
        assert linear_plan(rows, k, out, size)[0] == 4, (rows, k, out)                  # two rounds; wide tiles that fit badly


def test_ranges_of_k_of_short_products(linear_plan):
    for rows in (528, 584, 640):
        assert linear_plan(rows, 4096, 2560, 4) == (4, 4)
    for rows in (80, 104, 128):
        assert linear_plan(rows, 16384, 4096, 4) == (4, 16)                             # ranges of 2 KB of a row, not of 4
    assert linear_plan(112, 16448, 4096, 4) == (4, 8)


def test_orders_of_the_k_tiles_go_by_what_of_the_weights_the_chip_already_holds(linear_plan):
    lib = C.CDLL(iris_c_amd.LIB_PATH)
    lib.iris_hip_gemm_turns.argtypes = [C.c_long, C.c_size_t]
    turned = lambda wgs, mb: lib.iris_hip_gemm_turns(wgs, int(mb * (1 << 20))) == 3
    assert not turned(256, 4) and turned(256, 4.1) and turned(1, 4.1)                                 # one round: more than an L2
    assert not turned(257, 14) and turned(257, 14.1) and turned(5000, 14.1)                           # several


def test_partial_sums_beside_large_weights_are_stored_plainly(linear_plan):
    lib = C.CDLL(iris_c_amd.LIB_PATH)
    lib.iris_hip_gemm_tiles_plan.restype = C.c_float
    lib.iris_hip_gemm_tiles_plan.argtypes = [C.c_int] * 4 + [C.c_size_t] + [C.POINTER(C.c_int)] * 2

    def through(rows, k, out, size):
        shape, splits = C.c_int(), C.c_int()
        assert lib.iris_hip_gemm_tiles_plan(rows, out, k, size, 64 << 20, shape, splits) > 0 and splits.value > 1, (rows, k, out)
        return lib.iris_hip_gemm_tiles_through(shape, splits, rows, out, k)

    for rows, k, out, size in ((64, 9728, 2560, 4), (128, 9216, 3072, 4), (256, 4096, 2560, 4), (640, 3072, 3072, 4), (64, 12288, 3072, 4),
                               (90, 12288, 3072, 4), (72, 3072, 15360, 2), (100, 4096, 12288, 2), (128, 12288, 4096, 4)):
        assert through(rows, k, out, size) == 1, (rows, k, out)
    for rows, k, out, size in ((123, 12288, 3072, 4), (128, 6144, 6144, 4), (64, 3072, 15360, 2), (64, 2560, 19456, 2), (129, 2560, 19456, 2),
                               (64, 3072, 18432, 2), (64, 3072, 27648, 2), (128, 4096, 16384, 2), (100, 5120, 13824, 2), (100, 13824, 5120, 4),
                               (320, 12288, 3072, 4), (512, 9728, 2560, 4)):                          # the last two: more than 20 MB
        assert through(rows, k, out, size) == 0, (rows, k, out)
    assert lib.iris_hip_gemm_tiles_through(0, 1, 512, 2560, 9728) == 0                                # nothing to add


def test_projections_that_normalise_their_tiles_add_as_the_plain_layer_does(linear_plan):
    """Where the epilogue is taken, the plain layer is k_gemm_wide, k_gemm_dma, or tiles that take K whole, in one group and in order."""
    lib = C.CDLL(iris_c_amd.LIB_PATH)
    lib.iris_hip_gemm_tiles_plan.restype = C.c_float
    lib.iris_hip_gemm_tiles_plan.argtypes = [C.c_int] * 4 + [C.c_size_t] + [C.POINTER(C.c_int)] * 2
    seen = 0
    for heads in (8, 24, 32, 48, 100):
        for k in (64, 192, 320, 448, 512, 704, 1024, 2048, 2560, 4096):
            for out in range(256 * heads, 40000, 1408):
                for rows in list(range(300, 2000, 211)) + list(range(2000, 20000, 1117)):
                    if lib.iris_hip_linear_qknorm_plan(rows, k, out, 128 * heads, 128 * heads) != 1 or linear_plan(rows, k, out)[0] in (2, 3):
                        continue
                    shape, splits = C.c_int(), C.c_int()
                    lib.iris_hip_gemm_tiles_plan(rows, out, k, 2, 64 << 20, shape, splits)
                    assert lib.iris_hip_gemm_tiles_in_order(shape, splits, rows, out, k) == 1, (rows, k, out, heads)
                    seen += 1
    assert seen > 10


def test_projections_normalise_their_tiles_where_that_is_the_faster_form(linear_plan):
    lib = C.CDLL(iris_c_amd.LIB_PATH)
    plan = lambda rows, k, out, q, kv: lib.iris_hip_linear_qknorm_plan(rows, k, out, 128 * q, 128 * kv)
    assert linear_plan(4608, 3072, 27648) == (3, 256) and plan(4608, 3072, 27648, 24, 24) == 1       # the plain layer's own tiles
    for k in (64, 192, 448, 576):
        assert plan(4608, k, 9216, 24, 24) == 1
    for rows, k, out in ((320, 3072, 27648), (512, 3072, 9216), (2115, 192, 9216), (4608, 3072, 9216)):
        assert plan(rows, k, out, 24, 24) == 0
    assert plan(400000, 256, 6144, 24, 24) == 1          # more vectors than the norm kernel counts
    for rows, k, out, q, kv in ((255, 64, 768, 2, 2), (300, 72, 768, 2, 2), (300, 64, 800, 2, 2), (300, 64, 768, 4, 3), (300, 64, 768, 0, 0)):
        assert plan(rows, k, out, q, kv) == -1


# ------------------------------------------------------------------ the convolutions' kernel choice
FEW_IN, FEW_OUT, ONE_BY_ONE, THREE, THREE_HALF = 1, 2, 3, 4, 5


@pytest.fixture(scope="module")
def conv_plan():
    lib = C.CDLL(iris_c_amd.LIB_PATH)
    lib.iris_hip_conv2d_plan.argtypes = [C.c_void_p] * 3 + [C.c_int] * 8 + [C.POINTER(C.c_int)]
    lib.iris_hip_conv2d_plan.restype = None

    def call(h, w, cin, cout, k, stride=1, pb=0, pa=0, out=1 << 44, img=1 << 40, wt=1 << 46):
        """The addresses are only compared, never read."""
        p = (C.c_int * 2)()
        lib.iris_hip_conv2d_plan(out, img, wt, h, w, cin, cout, k, stride, pb, pa, p)
        return p[0]
    return call


@pytest.mark.parametrize("kernel,h,w,cin,cout,k,stride,pb,pa", [
    (FEW_IN, 512, 512, 3, 128, 3, 1, 1, 1), (FEW_OUT, 512, 512, 128, 3, 3, 1, 1, 1), (ONE_BY_ONE, 512, 512, 256, 128, 1, 1, 0, 0),
    (THREE, 256, 256, 128, 128, 3, 1, 1, 1), (THREE_HALF, 256, 256, 128, 128, 3, 2, 0, 1)])
def test_convolutions_whose_output_shares_memory_with_the_image_take_a_route_that_copies_it_first(conv_plan, kernel, h, w, cin, cout, k,
                                                                                                 stride, pb, pa):
    """The kernels that read the image directly store tiles whose surroundings other workgroups have still to read."""
    img = 1 << 40
    oh, ow = (h + pb + pa - k) // stride + 1, (w + pb + pa - k) // stride + 1
    in_bytes, out_bytes = h * w * cin * 4, oh * ow * cout * 4
    call = lambda out: conv_plan(h, w, cin, cout, k, stride, pb, pa, out=out, img=img)
    for out in (img, img + 16, img + in_bytes - 16, img - out_bytes + 16):
        assert call(out) == 0
    for out in (img + in_bytes, img - out_bytes, 1 << 44):
        assert call(out) == kernel


def test_few_output_channels_of_a_flat_image(conv_plan):
    """1 x 1 over all pixels as a column, the way a projection is called: tiles of 16 x 32 pixels would be almost empty."""
    assert conv_plan(65536, 1, 128, 3, 1) == conv_plan(262144, 1, 128, 16, 1) == conv_plan(1, 65536, 128, 28, 1) == ONE_BY_ONE
    assert conv_plan(65536, 1, 64, 3, 1) == 0
    assert conv_plan(65536, 1, 32, 3, 3, 1, 1, 1) == 0 and conv_plan(65536, 1, 128, 3, 3, 1, 1, 1) == FEW_OUT
    assert conv_plan(128, 128, 128, 28, 1) == ONE_BY_ONE and conv_plan(128, 128, 64, 28, 1) == 0
    for h, w in ((8, 8), (4096, 1), (100, 90), (512, 512), (1024, 1024)):
        assert conv_plan(h, w, 128, 3, 1) == conv_plan(h, w, 128, 3, 3, 1, 1, 1) == conv_plan(h, w, 64, 7, 2, 1, 0, 1) == FEW_OUT


def test_one_by_one_convolutions_of_few_pixels_and_many_channels_go_through_a_copy(conv_plan):
    for pixels in (256, 1000, 4096):
        for cin, cout in ((256, 64), (256, 128), (384, 100), (512, 32), (512, 128), (512, 256)):
            assert conv_plan(pixels, 1, cin, cout, 1) == 0, (pixels, cin, cout)
        for cout in (64, 128, 256):
            assert conv_plan(pixels, 1, 128, cout, 1) == ONE_BY_ONE
    assert conv_plan(16384, 1, 512, 128, 1) == 0
    for cin, cout in ((256, 64), (256, 128), (384, 100), (384, 256), (512, 32), (512, 128), (512, 256)):
        assert conv_plan(256, 256, cin, cout, 1) == conv_plan(512, 512, cin, cout, 1) == ONE_BY_ONE, (cin, cout)
    assert conv_plan(30000, 1, 256, 128, 1) == conv_plan(1000, 1, 256, 256, 1) == conv_plan(64, 1, 256, 128, 1) == ONE_BY_ONE


def test_three_by_three_convolutions_of_images_thinner_than_a_tile(conv_plan):
    three = lambda h, w, cin, cout, stride=1: conv_plan(h, w, cin, cout, 3, stride, 1, 1)
    for h, w in ((1, 4096), (4096, 1), (1, 20000), (20000, 1), (8, 3000), (3000, 8)):
        assert three(h, w, 512, 512) == three(h, w, 128, 384) == 0, (h, w)
    for cin, cout in ((64, 64), (64, 128), (128, 128), (256, 256), (512, 64), (1024, 1024)):
        assert three(1, 20000, cin, cout) == three(20000, 1, cin, cout) == 0, (cin, cout)
    assert three(4096, 1, 512, 512, 2) == three(20000, 1, 128, 128, 2) == three(1, 20000, 512, 512, 2) == 0
    # tiles that fit one round of the CUs, and images that fill theirs
    assert three(3, 1000, 512, 512) == three(1, 4096, 128, 128) == three(1000, 3, 256, 128) == THREE
    assert three(1, 4096, 512, 512, 2) == three(4096, 1, 256, 128, 2) == THREE_HALF
    for h, w in ((8, 8), (17, 17), (48, 48), (33, 500), (250, 130), (512, 512)):
        assert three(h, w, 512, 512) == three(h, w, 128, 64) == THREE and three(h, w, 256, 256, 2) == THREE_HALF, (h, w)


def test_few_input_channels_with_next_to_nothing_to_do_per_pixel(conv_plan):
    big = lambda cin, cout, k=1: conv_plan(1024, 1024, cin, cout, k, 1, k // 2, k // 2)
    for cin, cout, k in ((1, 1, 1), (1, 4, 1), (4, 4, 1), (16, 1, 1), (24, 1, 1), (1, 1, 3)):
        assert big(cin, cout, k) == 0, (cin, cout, k)
    assert big(32, 1) == big(32, 4) == FEW_OUT
    for cin, cout, k in ((3, 128, 3), (3, 3, 3), (2, 1, 3), (1, 2, 3), (8, 4, 1), (1, 32, 1), (32, 28, 1), (32, 512, 1)):
        assert big(cin, cout, k) == FEW_IN, (cin, cout, k)
    for h, w in ((16, 16), (256, 256)):
        assert conv_plan(h, w, 32, 128, 1) == conv_plan(h, w, 32, 512, 1) == 0
        assert conv_plan(h, w, 1, 1, 1) == conv_plan(h, w, 32, 4, 1) == conv_plan(h, w, 16, 512, 1) == conv_plan(h, w, 3, 128, 3, 1, 1, 1) == FEW_IN


@pytest.mark.parametrize("groups", [1, 2, 3, 8, 16])
def test_the_last_round_of_a_three_by_three_convolution_is_cut_into_ranges_that_cover_it_once(groups):
    share = C.CDLL(iris_c_amd.LIB_PATH).iris_hip_conv2d_share
    for total in (1, 2, 7, 8, 9, 31, 100, 255, 256, 257, 259, 288, 400, 511, 513, 1000, 1023, 2051):
        tiles = set()
        for xcd in range(8):
            shares = []
            for slot in range(32):
                s = (C.c_int * 5)()
                share(xcd, slot, total, groups, 0, s)
                shares.append(tuple(s))
            first, rest_first, rest = shares[0][:3]
            assert rest < 32 and (rest_first - first) % 32 == 0 and all(s[:3] == shares[0][:3] for s in shares)
            tiles |= set(range(first, rest_first + rest))
            at = 0
            for slot, (*_, u0, u1) in enumerate(shares):
                assert u0 == at and u1 - u0 <= groups and (u1 == u0 or (u1 - 1) // groups - u0 // groups <= 1)
                assert u1 > u0 or u0 == rest * groups                       # the workgroups that have a range come first
                for unit in range(u0, u1):
                    assert share(xcd, 0, total, groups, unit, (C.c_int * 5)()) == slot
                at = u1
            assert at == rest * groups
        assert tiles == set(range(total))


def test_the_last_round_is_cut_where_that_is_the_faster_form():
    cut = C.CDLL(iris_c_amd.LIB_PATH).iris_hip_conv2d_cut
    for oh, ow, cin, cout in CUT: assert cut(oh, ow, cin, cout) == 1, (oh, ow, cin, cout)
    for oh, ow, cin, cout in WHOLE: assert cut(oh, ow, cin, cout) == 0, (oh, ow, cin, cout)


CUT = [(64, 69, 512, 512), (64, 69, 512, 256), (122, 131, 512, 512), (177, 189, 512, 256), (16, 16, 512, 512)]
WHOLE = [(256, 256, 512, 512), (512, 512, 256, 256), (512, 512, 128, 128), (200, 200, 128, 128), (111, 119, 512, 512), (40, 40, 64, 64)]


# ------------------------------------------------------------------ row norms
def test_row_norms_take_a_wave_per_row_where_rows_are_many_and_short_and_a_workgroup_elsewhere():
    lib = C.CDLL(iris_c_amd.LIB_PATH)
    layer, rms, residual = 0, 1, 2
    workgroup, workgroup_reread, wave, wave_2048, wave_4096, wave_reread = range(6)
    plan = lambda kind, rows, dim, aligned=1: lib.iris_hip_row_norm_plan(kind, rows, dim, aligned)
    for kind in (layer, rms, residual):
        assert plan(kind, 1280, 64) == plan(kind, 1, 4096) == plan(kind, 20000, 3072) == workgroup
        assert plan(kind, 1281, 64) == plan(kind, 2047, 1024) == wave
        assert plan(kind, 3000, 1028) == plan(kind, 12800, 1536) == wave_2048
        assert plan(kind, 3000, 2052) == plan(kind, 4608, 3072) == workgroup
        assert plan(kind, 2048, 1023) == plan(kind, 2048, 1024, 0) == wave_reread
        assert plan(kind, 2047, 1023) == plan(kind, 4608, 3071) == plan(kind, 4608, 3072, 0) == plan(kind, 512, 5120) == workgroup_reread
    assert plan(layer, 3000, 2048) == plan(rms, 3000, 2048) == wave_2048 and plan(residual, 3000, 1540) == workgroup
    assert plan(layer, 32768, 2052) == wave_4096 and plan(rms, 32768, 2052) == plan(residual, 32768, 2052) == workgroup
    assert plan(layer, 32768, 5120) == wave_reread and plan(rms, 32768, 5120) == workgroup_reread


def test_profile_summaries_say_which_source_they_were_taken_on():
    """Every summary under profiles/ names the commit and the hash of the kernel source it was measured on, and
    bench.py can tell from the C2 counter file whether its traffic figure belongs to the kernel source in the tree."""
    import glob
    import os
    import re
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    files = sorted(glob.glob(os.path.join(root, "profiles", "*.txt")))
    assert len(files) >= 10
    for path in files:
        text = open(path).read()
        assert re.search(r"^taken_on_commit: [0-9a-f]{40}$", text, re.M), path
        assert re.search(r"^kernel_source_sha256: [0-9a-f]{16}\s+\(iris_c_amd/csrc/\w+\.hip\)$", text, re.M), path
    sys.path.insert(0, root)
    import bench
    nbytes, source, stale = bench.traffic_on_file()
    assert nbytes and nbytes > 113_246_208 and source.endswith("hbm_traffic.txt") and stale in (True, False)


# ------------------------------------------------------------------ group norm as one launch
@pytest.fixture(scope="module")
def norm_plan():
    return C.CDLL(iris_c_amd.LIB_PATH).iris_hip_group_norm_plan


def test_group_norm_is_one_launch_only_where_all_its_workgroups_find_a_cu(norm_plan):
    for hw, c in ((1 << 20, 128), (512 * 512, 256), (128 * 128, 512)):
        assert norm_plan(hw, c, 32, 256) == norm_plan(hw, c, 32, 304) == 1
        for cus in (0, 32, 64, 128, 255):
            assert norm_plan(hw, c, 32, cus) == 0


def test_group_norm_is_one_launch_for_the_shapes_it_takes(norm_plan):
    for c, groups, takes in ((128, 32, 1), (64, 8, 1), (2048, 64, 1), (128, 4, 0), (96, 8, 0), (512, 128, 0), (64, 32, 0), (4096, 32, 0), (130, 32, 0)):
        assert norm_plan((64 << 20) // (4 * c), c, groups, 256) == takes, (c, groups)
    assert norm_plan((1 << 28) // 32, 128, 32, 256) == 0 and norm_plan((1 << 28) // 32 - 1, 128, 32, 256) == 1     # 4 GiB
    assert norm_plan(100, 128, 32, 256) == 0


def test_group_norm_is_one_launch_from_ten_megabytes_on(norm_plan):
    for c in (128, 256, 512):
        n = (10 << 20) // (4 * c)
        assert norm_plan(n, c, 32, 256) == 1 and norm_plan(n - 1, c, 32, 256) == 0
