"""GPU parity of the decode attention's key ranges (needs an MI355X): ranges are
cut on the device from each sequence's own length, a short sequence keeps one,
and the last workgroup to arrive merges them in batches.  Lengths sit at the
edges of a wave's 16-key block, of a range, of the one-range limit (384 keys)
and of the planned length; the counts at the edges of a merge batch (8 and 16).

Bound as in test_gpu_attn.py: 2^-8 * (sum p|v| / sum p + |exact|).  Cache rows
past a sequence's end hold NaN: a row that no query may see must not be used.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from starter_amd import kernels as K
from tests._util import BF16, bits, randn_bf16
from tests.test_gpu_attn import _check_attention
from tests.test_gpu_attn_rope import _assert_same, _fused, _setup, _unfused

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
D = 128


@pytest.mark.parametrize("B,R,HQ,HKV,cap,maxlen,nsplit,starts,shift", [
    (8, 1, 8, 2, 640, 640, 5, (0, 15, 16, 127, 382, 383, 384, 639), 0),   # one-range limit: 384 and 385 keys
    (3, 1, 8, 2, 4300, 4300, 33, (2111, 4223, 4299), 1),                 # 17, 33 and 34 grains of 64: batches of 16 and a rest
    (2, 2, 8, 2, 1200, 1200, 9, (511, 1150), 1),                         # 8 rows, 4 and 9 ranges, 2-byte aligned output
    (2, 5, 8, 2, 1200, 1200, 9, (380, 1194), 0),                         # two row blocks
    (1, 16, 8, 2, 2300, 2300, 17, (2270,), 1),                           # four row blocks, more than 16 ranges
    (70, 1, 4, 4, 500, 500, 2, tuple(7 * b for b in range(70)), 0),      # more sequences than lanes
    (2, 1, 32, 8, 5000, 5000, None, (400, 4999), 0),                     # the planned split, far and near
])
def test_key_ranges_match_oracle(B, R, HQ, HKV, cap, maxlen, nsplit, starts, shift):
    g = torch.Generator().manual_seed(B * 100 + R)
    q = randn_bf16((B, HQ, R, D), 1.0, g)
    kc = randn_bf16((B, HKV, cap, D), 1.0, g)
    vc = randn_bf16((B, HKV, cap, D), 1.0, g)
    pos = np.array(starts, np.int32)
    ref = oracle.decode_attention(bits(q), bits(kc), bits(vc), pos, D ** -0.5, with_abs=True)
    for b in range(B):
        kc[b, :, starts[b] + R:] = float("nan")
        vc[b, :, starts[b] + R:] = float("nan")
    attn = K.DecodeAttention(B, HQ, HKV, D, cap, DEV, R=R, maxlen=maxlen, nsplit=nsplit)
    buf = torch.zeros(B * R * HQ * D + 8, dtype=BF16, device=DEV)
    out = buf[shift:shift + B * R * HQ * D].view(B, R, HQ, D)
    qd, kd, vd, pd = q.to(DEV), kc.to(DEV), vc.to(DEV), torch.from_numpy(pos).to(DEV)
    for _ in range(2):   # the arrival counters are back at zero
        attn(qd, kd, vd, pd, out)
        torch.cuda.synchronize()
        _check_attention(out, ref, f"ranges B={B} R={R}")
    assert not bool((buf[:shift] != 0).any()) and not bool((buf[shift + out.numel():] != 0).any())


@pytest.mark.parametrize("B,R,cap,nsplit,starts", [
    (4, 1, 1500, 8, (383, 384, 1023, 1100)),   # the new row starts a range, a block, or lies inside one
    (2, 3, 900, 7, (382, 765)),                # new rows on both sides of the one-range limit and of a range edge
    (70, 1, 300, 2, tuple(4 * b for b in range(70))),
])
def test_fused_rows_at_range_edges(B, R, cap, nsplit, starts):
    """The first key block is requested before the new rows are written, unless
    it holds them: the fused launch equals rotary step, then attention."""
    eps = 1e-6
    qkv, qw, kw, cos, sin, kc, vc, pos = _setup(B, 8, 2, R, cap, starts, seed=B + R)
    attn = K.DecodeAttention(B, 8, 2, D, cap, DEV, nsplit=nsplit, R=R)
    kc2, vc2 = kc.clone(), vc.clone()
    ref = _unfused(attn, qkv, qw, kw, cos, sin, pos, kc, vc, eps)
    out = _fused(attn, qkv, qw, kw, cos, sin, pos, kc2, vc2, eps)
    torch.cuda.synchronize()
    _assert_same(kc2, kc, "k cache")
    _assert_same(vc2, vc, "v cache")
    _assert_same(out, ref, "attention output")
