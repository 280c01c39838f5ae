"""Attention of head_dim 128 whose workgroups give the two tiles of a group to two halves of their waves (k_fa_fwd_hd128 with
PARTS = 2: 197 - 640 rows of 24 heads), against the oracle at the bar of the other attention tests: odd and even numbers of tiles,
waves and tiles without queries or keys. The same sizes with a key mask, which keep one wave to its queries: valid keys in some
tiles only, no valid key at all."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from gpu_harness import Dev, assert_parity

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return Dev()


def call(dev, orc, heads, kv, seq_q, seq_k, causal, mask, amp=1.0):
    rng = np.random.default_rng(seq_q * 31 + seq_k + heads)
    q, kvd = heads * 128, kv * 128
    ldi, rows = q + 2 * kvd, max(seq_q, seq_k)
    buf = O.f32_to_bf16((rng.standard_normal((rows, ldi)) * amp).astype(np.float32))
    scale = 128 ** -0.5
    route = (C.c_int * 6)()
    dev.lib.iris_hip_fa_hd128_route(seq_q, seq_k, heads, int(causal), int(mask is not None), route)
    assert route[0] == 0 and route[5] == (2 if mask is None else 1)
    out, kernel = dev.attention(buf, ldi, 0, q, q + kvd, seq_q, seq_k, heads, kv, 128, scale, causal, mask)
    assert kernel == "fa_hd128"
    want = orc.attention_bf16(buf, ldi, 0, q, q + kvd, seq_q, seq_k, heads, kv, 128, scale, causal, mask)
    return O.bf16_to_f32(out[:, :q]), want


# 2 x 2 waves (workgroups of 32 queries), then 4 x 2 (64 queries)
@pytest.mark.parametrize("heads,kv,seq_q,seq_k", [(24, 24, 197, 197), (24, 24, 300, 256), (24, 8, 320, 257), (24, 24, 320, 320), (32, 8, 255, 384),
                                                  (24, 24, 385, 385), (30, 10, 512, 512), (24, 12, 513, 449), (24, 24, 640, 640)])
@pytest.mark.parametrize("causal", [False, True])
def test_against_the_oracle(dev, orc, heads, kv, seq_q, seq_k, causal):
    got, want = call(dev, orc, heads, kv, seq_q, seq_k, causal, None)
    assert_parity(got, want, f"{heads} x {seq_q} x {seq_k}")


@pytest.mark.parametrize("seq", [320, 449])
@pytest.mark.parametrize("valid", ["first", "second_tile", "third_and_last", "prefix", "random"])
def test_masks(dev, orc, seq, valid):
    mask = np.zeros(seq, np.int32)
    if valid == "first": mask[0] = 1
    if valid == "second_tile": mask[64:128] = 1
    if valid == "third_and_last": mask[130:150] = mask[-1:] = 1
    if valid == "prefix": mask[:201] = 1
    if valid == "random": mask[np.random.default_rng(seq).random(seq) < 0.3] = 1
    got, want = call(dev, orc, 24, 24, seq, seq, False, mask)
    assert_parity(got, want, valid)


@pytest.mark.parametrize("seq", [320, 449])
def test_no_valid_key_gives_zero_rows(dev, orc, seq):
    got, _ = call(dev, orc, 24, 24, seq, seq, False, np.zeros(seq, np.int32))
    assert not got.any()


@pytest.mark.parametrize("seq", [320, 512])
def test_large_scores(dev, orc, seq):
    """Scores up to some hundreds: the halves' maxima differ by far more than the range of their sums."""
    got, want = call(dev, orc, 24, 24, seq, seq, False, None, amp=6.0)
    assert_parity(got / 6.0, want / 6.0, "large scores")
