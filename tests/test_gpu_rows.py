"""The 16-byte row kernels of prefill (SwiGLU, q/k norm + rotary step + cache write) on an MI355X.

Operands that are 16-byte aligned with strides of 8 elements take the vector
kernels, everything else the one-element ones; both must give the same bits,
and SwiGLU the oracle's.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from starter_amd import kernels as K
from tests._util import BF16, bits, randn_bf16
from tests.test_oracle import rope_tables_cpu

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
D = 128


def _shifted(t: torch.Tensor, by: int, pad: int = 0) -> torch.Tensor:
    """A copy of t [rows, cols] whose base lies `by` elements past an aligned address and whose rows are `pad` wider."""
    rows, cols = t.shape
    buf = torch.full((rows * (cols + pad) + by,), float("nan"), dtype=BF16, device=DEV)
    v = buf[by:].view(rows, cols + pad)[:, :cols]
    return v.copy_(t.to(DEV))


@pytest.mark.parametrize("M,I", [(1, 8), (3, 2048), (5, 2056), (1030, 264), (2, 9728), (7, 12), (4, 9)])
def test_swiglu_forms_equal_the_oracle(M, I):
    g = torch.Generator().manual_seed(M + I)
    gu = randn_bf16((M, 2 * I), 3.0, g)
    special = torch.tensor([float("inf"), float("-inf"), float("nan"), 0.0, -0.0, 88.0, -88.0, 3e38]).to(BF16)
    gu[0, :min(8, I)] = special[:min(8, I)]
    want = oracle.swiglu(bits(gu))
    for by, pad in ((0, 0), (0, 8), (8, 0), (1, 0), (0, 3)):
        src = _shifted(gu, by, pad)
        for oby, opad in ((0, 0), (0, 5), (4, 0)):
            out = torch.full((M * (I + opad) + oby,), 7.0, dtype=BF16, device=DEV)
            view = out[oby:].view(M, I + opad)[:, :I]
            K.swiglu(src, out=view)
            torch.cuda.synchronize()
            got = bits(view)
            nan = (want & 0x7FFF) > 0x7F80
            assert np.array_equal(got[~nan], want[~nan]) and np.all((got[nan] & 0x7FFF) > 0x7F80), (by, pad, oby, opad)
            assert (out[oby:].view(M, I + opad)[:, I:] == 7.0).all()


@pytest.mark.parametrize("M,I", [(65535 + 9, 2048), (700, 8), (513, 16), (129, 72), (3, 1032), (1000, 1016)])
def test_swiglu_of_every_row_packing(M, I):
    """1 to 256 threads per row, part of them idle, a last workgroup with fewer
    rows, and more rows than the grid has."""
    g = torch.Generator().manual_seed(M + I)
    gu = randn_bf16((M, 2 * I), 3.0, g)
    assert np.array_equal(bits(K.swiglu(gu.to(DEV))), oracle.swiglu(bits(gu)))


@pytest.mark.parametrize("M", [4, 17, 64])
def test_swiglu_of_few_rows_is_no_slower_in_16_byte_accesses(M):
    """The vector kernel against the one-element kernel (which an odd output
    stride selects) where launch and latency decide: a thread must not work
    through several rows while most of the chip is idle (that took 1.2 to 1.8
    times as long here)."""
    I, reps = 9728, 200   # (one replay of 0.5 ms: its launch, which may vary by 5 us, does not count)
    gu = torch.randn(M, 2 * I, device=DEV).to(BF16)

    def best(out):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            K.swiglu(gu, out=out)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(reps):
                K.swiglu(gu, out=out)
        times = []
        for _ in range(20):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            graph.replay()
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    scalar = best(torch.empty((M, I + 1), dtype=BF16, device=DEV)[:, :I])
    assert best(torch.empty((M, I), dtype=BF16, device=DEV)) < 1.15 * scalar


@pytest.mark.parametrize("B,T,HQ,HKV,cap,tree", [
    (2, 33, 32, 8, 128, False), (3, 1, 4, 2, 64, False), (1, 5, 5, 1, 20, True), (2, 8, 8, 2, 40, True),
    (1, 300, 3, 3, 256, False),   # rows past the cache and past the table are skipped
    (50, 8, 5, 1, 300, True), (4, 1, 200, 28, 64, False), (1, 342, 1, 1, 400, True),   # from 1024 heads on 16-byte rows
    (1, 341, 1, 1, 400, False)])                                                      # the most that take the other kernel
def test_rope_vector_rows_equal_scalar_rows(B, T, HQ, HKV, cap, tree):
    g = torch.Generator().manual_seed(B * T)
    W = (HQ + 2 * HKV) * D
    cos, sin = (t.to(DEV) for t in rope_tables_cpu(D, 1e6, cap + 4))
    qkv = randn_bf16((B * T, W), 1.0, g)
    qw, kw = ((1 + 0.1 * torch.randn(D, generator=g)).to(BF16).to(DEV) for _ in range(2))
    pos = torch.tensor([3 + 5 * b for b in range(B)], dtype=torch.int32, device=DEV)
    depth = torch.tensor([t // 2 for t in range(T)], dtype=torch.int32, device=DEV) if tree else None
    outs = []
    for by, pad in ((0, 0), (0, 16), (1, 0), (0, 2)):   # two aligned forms, two that are not
        q = torch.full((B, HQ, T, D), 5.0, dtype=BF16, device=DEV)
        kc, vc = (torch.full((B, HKV, cap, D), 6.0, dtype=BF16, device=DEV) for _ in range(2))
        K.qk_norm_rope_cache(_shifted(qkv, by, pad), qw, kw, cos, sin, pos, q, kc, vc, T, 1e-6, depth=depth)
        torch.cuda.synchronize()
        outs.append((q, kc, vc))
    for o in outs[1:]:
        for a, b in zip(o, outs[0]):
            assert torch.equal(a.view(torch.int16), b.view(torch.int16))
