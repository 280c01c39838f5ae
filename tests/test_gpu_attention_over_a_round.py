"""Attention of head_dim 128 in grids of a few more 128-query workgroups than CUs, where the kernel changes (without causal) or
stays (causal, the last workgroups in a second round), against attention in 32 bits."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle as O
from gpu_harness import Dev, assert_parity

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return Dev()


def reference(buf, seq, heads, kv, causal, mask):
    x = torch.from_numpy(O.bf16_to_f32(buf)).cuda()
    q, k, v = x.split([heads * 128, kv * 128, kv * 128], 1)
    out = torch.empty(seq, heads, 128, device="cuda")
    hidden = torch.zeros(seq, seq, dtype=torch.bool, device="cuda")
    if causal: hidden |= torch.ones_like(hidden).triu(1)
    if mask is not None: hidden |= torch.from_numpy(mask == 0).cuda()
    for h in range(heads):
        col = slice(128 * (h * kv // heads), 128 * (h * kv // heads) + 128)
        s = q[:, 128 * h:128 * h + 128].contiguous() @ k[:, col].T.contiguous() * 128 ** -0.5
        out[:, h] = torch.softmax(s.masked_fill(hidden, -float("inf")), 1) @ v[:, col].contiguous()
    return out.view(seq, -1).cpu().numpy()


@pytest.mark.parametrize("heads,kv,seq,causal,valid,kind,waves,blocks", [
    (24, 24, 1281, 0, None, 1, 8, 2), (24, 8, 1360, 0, 1300, 1, 8, 2), (30, 30, 1025, 0, 65, 1, 8, 2), (30, 30, 1088, 0, None, 1, 8, 2),
    (24, 24, 1361, 1, None, 0, 8, 1), (32, 8, 1025, 1, 118, 0, 4, 1), (32, 8, 1152, 1, 1152, 0, 4, 1), (32, 8, 1536, 1, None, 0, 8, 1),
    (24, 24, 1536, 1, 500, 0, 4, 1), (16, 16, 2049, 1, 200, 0, 8, 1), (32, 8, 1153, 1, 700, 0, 8, 2), (32, 8, 1537, 1, None, 0, 8, 2)])
def test_against_32_bits(dev, heads, kv, seq, causal, valid, kind, waves, blocks):
    plan = (C.c_int * 6)()
    dev.lib.iris_hip_fa_hd128_route(seq, seq, heads, causal, int(valid is not None), plan)
    assert (plan[0], plan[1], plan[2]) == (kind, waves, blocks)
    q, ld = heads * 128, (heads + 2 * kv) * 128
    buf = O.f32_to_bf16(np.random.default_rng(seq).standard_normal((seq, ld)).astype(np.float32))
    mask = (np.arange(seq) < valid).astype(np.int32) if valid is not None else None
    out, kernel = dev.attention(buf, ld, 0, q, q + kv * 128, seq, seq, heads, kv, 128, 128 ** -0.5, bool(causal), mask)
    assert kernel == "fa_hd128"
    assert_parity(O.bf16_to_f32(out), reference(buf, seq, heads, kv, causal, mask), f"{heads} x {seq}")
