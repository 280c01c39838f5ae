"""Attention of head_dim 128 in grids of 256-query workgroups with 64-query ones behind them (a few workgroups more than whole
rounds of the CUs), against attention in 32 bits: tails of one query, of a whole and of one more than a whole workgroup, even and
odd numbers of key tiles, key masks that end the walk early, and Q normalised on the way in."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle as O
from gpu_harness import Dev, assert_parity

pytestmark = pytest.mark.gpu
HEADS, KV = 64, 8


@pytest.fixture(scope="module")
def dev():
    return Dev()


def route(dev, seq_q, seq_k, masked):
    plan = (C.c_int * 6)()
    dev.lib.iris_hip_fa_hd128_route(seq_q, seq_k, HEADS, 0, int(masked), plan)
    return plan


def rows(n):
    rng = np.random.default_rng(n)
    return O.f32_to_bf16(rng.standard_normal((n, (HEADS + 2 * KV) * 128)).astype(np.float32))


def reference(buf, seq_q, seq_k, mask):
    x = torch.from_numpy(O.bf16_to_f32(buf)).cuda()
    q = x[:seq_q, :HEADS * 128].view(seq_q, HEADS, 128)
    k, v = (x[:seq_k, (HEADS + i * KV) * 128:(HEADS + (i + 1) * KV) * 128].view(seq_k, KV, 128) for i in (0, 1))
    out = torch.empty(seq_q, HEADS, 128, device="cuda")
    for h in range(HEADS):
        s = q[:, h].contiguous() @ k[:, h * KV // HEADS].T.contiguous() * 128 ** -0.5
        if mask is not None: s[:, torch.from_numpy(mask).cuda() == 0] = -float("inf")
        out[:, h] = torch.softmax(s, 1) @ v[:, h * KV // HEADS].contiguous()
    return out.view(seq_q, -1).cpu().numpy()


@pytest.mark.parametrize("seq_q,seq_k,valid", [(1025, 1025, None), (1088, 961, None), (1089, 1040, None), (1151, 1151, None), (1216, 1217, 1217),
                                               (1100, 1100, 700), (1100, 1153, 65), (1089, 1089, 1)])
def test_against_32_bits(dev, seq_q, seq_k, valid):
    plan = route(dev, seq_q, seq_k, valid is not None)
    assert plan[0] == 3 and 256 * plan[3] + 64 * plan[4] >= seq_q > 256 * plan[3] + 64 * (plan[4] - 1)
    buf = rows(max(seq_q, seq_k))
    mask = (np.arange(seq_k) < valid).astype(np.int32) if valid is not None else None
    q = HEADS * 128
    out, kernel = dev.attention(buf, q + 2 * KV * 128, 0, q, q + KV * 128, seq_q, seq_k, HEADS, KV, 128, 128 ** -0.5, False, mask)
    assert kernel == "fa_hd128"
    assert_parity(O.bf16_to_f32(out), reference(buf, seq_q, seq_k, mask), f"{seq_q} x {seq_k}")


@pytest.mark.parametrize("hidden", ["the first tile", "even tiles", "odd tiles", "all but the last key", "the first of each tile"])
@pytest.mark.parametrize("seq_q,seq_k", [(1089, 1089), (1100, 1153)])
def test_masks_that_hide_all_that_one_of_two_waves_has_taken_so_far(dev, seq_q, seq_k, hidden):
    """Two waves take the tiles of 64 keys in turn: one may have met no valid key yet, or none at all, when they merge."""
    assert route(dev, seq_q, seq_k, True)[0] == 3
    key = np.arange(seq_k)
    mask = {"the first tile": key >= 64, "even tiles": key // 64 % 2 == 1, "odd tiles": key // 64 % 2 == 0, "all but the last key": key == seq_k - 1,
            "the first of each tile": key % 64 != 0}[hidden].astype(np.int32)
    buf, q = rows(max(seq_q, seq_k)), HEADS * 128
    out, kernel = dev.attention(buf, q + 2 * KV * 128, 0, q, q + KV * 128, seq_q, seq_k, HEADS, KV, 128, 128 ** -0.5, False, mask)
    assert kernel == "fa_hd128"
    assert_parity(O.bf16_to_f32(out), reference(buf, seq_q, seq_k, mask), f"{seq_q} x {seq_k}, {hidden} hidden")


def test_no_valid_key_gives_zero_rows(dev):
    assert route(dev, 1089, 1089, True)[0] == 3
    q = HEADS * 128
    out, _ = dev.attention(rows(1089), q + 2 * KV * 128, 0, q, q + KV * 128, 1089, 1089, HEADS, KV, 128, 128 ** -0.5, False, np.zeros(1089, np.int32))
    assert not out.any()


def test_q_normalised_on_the_way_in_gives_the_bits_of_the_two_calls(dev):
    seq, q, ld = 1100, HEADS * 128, (HEADS + 2 * KV) * 128
    assert route(dev, seq, seq, False)[0] == 3
    rng = np.random.default_rng(5)
    buf, w = rows(seq), rng.standard_normal(128).astype(np.float32)
    ang = rng.uniform(-3, 3, (seq, 64)).astype(np.float32)
    cos, sin = np.cos(ang), np.sin(ang)
    got, kernel, _ = dev.attention_qnorm(buf, ld, 0, q, q + KV * 128, seq, seq, HEADS, KV, 128, 128 ** -0.5, w, cos, sin, 1e-6, 0)
    assert kernel == "fa_hd128_qnorm"
    normed = dev.norm_rope(buf, ld, 0, w, cos, sin, seq, HEADS, 128, 1e-6, 0)
    want, _ = dev.attention(normed, ld, 0, q, q + KV * 128, seq, seq, HEADS, KV, 128, 128 ** -0.5)
    assert np.array_equal(got, want)
