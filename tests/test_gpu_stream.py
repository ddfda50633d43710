"""GPU parity of the stream path (SK_PATH_STREAM, csrc/sk_stream.hpp) against the CPU oracle (needs an MI355X).

Weight and activation rows are loaded straight into LDS rings; the waves of a
workgroup form K groups and, above 16 rows, share a group's rows.  Checked at
the edges of every wave shape's rows, with tiles that leave rows of their
last slab unused, a ragged N, K slices of unequal and of very few units
(fewer than the ring is deep), split-K finishes, the SwiGLU pairing of a tile
whose halves do not fill whole slabs, strided operands, and the residual
producer.
"""

from __future__ import annotations

import pytest
import torch

import oracle
from starter_amd import _lib
from starter_amd import kernels as K
from starter_amd._lib import SK_ERR_CONFIG, SK_OK, SK_PATH_STREAM, SkConfig
from tests._util import BF16, assert_gateup_parity, assert_parity, bits, from_bits, randn_bf16

DEV = "cuda:0"


def stream(rows, split=1, mg=1, ku=2):
    """Four waves: 4 / mg K groups of mg waves, units of 32 ku columns."""
    return SkConfig.make(SK_PATH_STREAM, waves=4, ku=ku, rows=rows, split=split, groups=mg)


def _ids(c):
    return f"r{c.rows}-s{c.split}-mg{c.groups}-ku{c.ku}"


# (N, K, config, row counts)
GEMM_CASES = [
    (2560, 9728, stream(32, 3), (1, 3, 16)),
    (6144, 2560, stream(24), (2, 15, 16)),
    (777, 2560, stream(10), (5, 16)),              # ragged N, 6 rows of the slab unused
    (777, 128, stream(80), (1, 16)),               # two units: fewer than the K groups
    (1000, 640, stream(33, 3), (7,)),              # ten units in slices of 4, 4, 2; odd tile rows
    (2560, 9728, stream(40, 4, 2), (17, 33, 64)),
    (777, 320, stream(48, 1, 2), (1, 32, 40)),     # five units for two K groups
    (1000, 192, stream(20, 3, 2), (50,)),          # one unit per slice: the second K group has none
    (6144, 2560, stream(24, 1, 2, 4), (49, 64)),
    (6144, 2560, stream(24, 1, 4, 4), (65, 100, 128)),
    (777, 384, stream(70, 1, 4, 4), (128,)),       # three 128-column units
    (1000, 1280, stream(64, 4, 4, 4), (97,)),      # slices of 3, 3, 3, 1 units
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", GEMM_CASES, ids=lambda c: f"{c[0]}x{c[1]}-{_ids(c[2])}")
def test_stream_gemm(case):
    N, Kd, cfg, ms = case
    g = torch.Generator().manual_seed(N + Kd + cfg.rows)
    w = randn_bf16((N, Kd), 0.02, g)
    wd = w.to(DEV)
    for M in ms:
        x = randn_bf16((M, Kd), 1.0, g)
        # rows of a wider matrix (row stride > K, odd multiple of 8)
        xd = torch.full((M, Kd + 24), float("nan"), dtype=BF16, device=DEV)[:, :Kd]
        xd.copy_(x)
        out = torch.full((M, N + 3), float("nan"), dtype=BF16, device=DEV)
        ws = K._workspace(K.SK_OP_GEMM, M, N, Kd, cfg, DEV)
        ref = from_bits(oracle.gemm(bits(x), bits(w)))
        for _ in range(2):   # the second call finds the counters back at zero
            K.gemm(xd, wd, out=out[:, :N], config=cfg, ws=ws)
            torch.cuda.synchronize()
            assert_parity(out[:, :N], ref, f"N={N} K={Kd} {cfg} M={M}")
        assert torch.isnan(out[:, N:]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("I,Kd,cfg,M", [
    (9728, 2560, stream(38, 1, 2), 17), (9728, 2560, stream(38, 1, 2), 64), (9728, 2560, stream(40, 1, 4, 4), 128),
    (1000, 2560, stream(19), 16),                  # halves of 19 rows: the up rows start at row 24
    (1000, 256, stream(33, 1, 2), 40), (500, 384, stream(13, 1, 4, 4), 77)], ids=str)
def test_stream_gateup(I, Kd, cfg, M):
    g = torch.Generator().manual_seed(I + M)
    wgu, x = randn_bf16((2 * I, Kd), 0.02, g), randn_bf16((M, Kd), 1.0, g)
    wd = wgu.to(DEV)
    out = K.gateup_swiglu(x.to(DEV), wd[:I], wd[I:], config=cfg)
    torch.cuda.synchronize()
    assert_gateup_parity(out, bits(x), bits(wgu[:I]), bits(wgu[I:]), f"I={I} {cfg} M={M}")


@pytest.mark.gpu
@pytest.mark.parametrize("N,Kd,cfg,M", [
    (2560, 9728, stream(32, 3), 16), (2560, 4096, stream(32, 3, 2), 33), (2560, 4096, stream(16, 1, 4, 4), 128),
    (200, 512, stream(48, 2, 2), 20)], ids=str)
def test_stream_residual_producer(N, Kd, cfg, M):
    """xout equals bf16(r + y) with y of the same plan bit for bit, and the
    group sums equal the fp64 sums of xout^2 (16 fp32 squares added pairwise:
    within 8 roundings)."""
    g = torch.Generator().manual_seed(N + M)
    a, w, r = (randn_bf16(s, c, g).to(DEV) for s, c in (((M, Kd), 1.0), ((N, Kd), 0.02), ((M, N), 1.0)))
    y = K.gemm(a, w, config=cfg)
    ro, sq = torch.empty_like(r), torch.full((M, K.sumsq_groups(M, N)), float("nan"), device=DEV)
    K.gemm_residual(a, w, r, ro, sq, config=cfg)
    want = (r.float() + y.float()).to(BF16)
    assert torch.equal(ro, want)
    padded = torch.zeros((M, 16 * sq.shape[1]), dtype=torch.float64, device=DEV)
    padded[:, :N] = want.double()
    assert torch.allclose(sq.double(), padded.pow(2).view(M, -1, 16).sum(-1), rtol=8 * 2.0 ** -24, atol=0)


# Persistent tiles: workgroups with unequal slabs, a ragged last slab, last
# tiles of one slab, fewer units than the ring is deep, odd unit counts (the
# fragment registers swap roles from tile to tile) and more workgroups asked
# for than there are slabs.
TILES_CASES = [(777, 64, 3, 1), (777, 128, 3, 64), (777, 320, 2, 65), (2577, 192, 16, 128), (1000, 2560, 4, 100),
               (50, 384, 256, 33), (41001, 320, 256, 17)]


def tiles(grid):
    return SkConfig.make(SK_PATH_STREAM, waves=8, ku=2, rows=160, split=1, grid=grid, groups=4)


@pytest.mark.gpu
@pytest.mark.parametrize("N,Kd,grid,M", TILES_CASES)
def test_stream_persistent_tiles(N, Kd, grid, M):
    g = torch.Generator().manual_seed(N + Kd + M)
    w, x = randn_bf16((N, Kd), 0.02, g), randn_bf16((M, Kd), 1.0, g)
    wide = torch.full((N, Kd + 40), float("nan"), dtype=BF16, device=DEV)
    wide[:, :Kd] = w.to(DEV)
    xd = torch.full((M, Kd + 24), float("nan"), dtype=BF16, device=DEV)[:, :Kd]
    xd.copy_(x)
    ref = from_bits(oracle.gemm(bits(x), bits(w)))
    for pad in (0, 3):   # 8-byte aligned output rows or not (with an odd N)
        out = torch.full((M, (N + 7) // 4 * 4 + pad), float("nan"), dtype=BF16, device=DEV)
        K.gemm(xd, wide[:, :Kd], out=out[:, :N], config=tiles(grid))
        torch.cuda.synchronize()
        assert_parity(out[:, :N], ref, f"N={N} K={Kd} grid={grid} M={M}")
        assert torch.isnan(out[:, N:]).all()
    # the fused argmax: of this kernel's own logits, the lowest index of ties
    ws = K._workspace(K.SK_OP_LM_ARGMAX, M, N, Kd, tiles(grid), DEV)
    for _ in range(2):
        ids, maxv = K.lm_argmax(xd, wide[:, :Kd], config=tiles(grid), ws=ws)
        logits = out[:, :N].float()
        best = logits.max(-1).values
        first = (logits == best[:, None]).float().argmax(-1)
        assert torch.equal(maxv, best) and torch.equal(ids, first)


@pytest.mark.gpu
@pytest.mark.parametrize("N,Kd,M", [(40960, 320, 33), (41000, 128, 64), (45001, 640, 65), (40960, 192, 130)])
def test_default_routes_of_many_weight_rows(N, Kd, M):
    g = torch.Generator().manual_seed(N + M)
    w, x = randn_bf16((N, Kd), 0.02, g).to(DEV), randn_bf16((M, Kd), 1.0, g).to(DEV)
    mm = K.SkinnyMatmul(M, N, Kd, DEV)
    out = mm(x, w)
    assert_parity(out, (x.float() @ w.float().t()).cpu(), "fp32 product")
    am = K.LmArgmax(M, N, Kd, DEV)
    ids, maxv = am(x, w)
    ids, maxv = ids.clone(), maxv.clone()
    best = out.float().max(-1).values
    assert torch.equal(maxv[:128], best[:128])
    assert torch.equal(ids[:128], (out[:128].float() == best[:128, None]).float().argmax(-1))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        mm(x, w), am(x, w)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        c_out, (c_ids, c_max) = mm(x, w), am(x, w)
    for _ in range(3):
        c_out.zero_(), c_ids.zero_(), c_max.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c_out, out) and torch.equal(c_ids, ids) and torch.equal(c_max, maxv)


# Calls without a configuration take the stream plan that their workspace
# allows: every route of a shape against the oracle, also replayed from a graph.
ROUTES = [(6144, 2560, m) for m in (2, 16, 17, 48, 49, 64, 65, 128, 130)] + \
         [(2560, 4096, m) for m in (16, 17, 64, 96, 97, 128)] + \
         [(2560, 9728, m) for m in (2, 3, 16, 17, 64, 65, 128)]


@pytest.mark.gpu
@pytest.mark.parametrize("N,Kd,M", ROUTES)
def test_default_routes(N, Kd, M):
    g = torch.Generator().manual_seed(N + M)
    w, x = randn_bf16((N, Kd), 0.02, g), randn_bf16((M, Kd), 1.0, g)
    wd, xd = w.to(DEV), x.to(DEV)
    ref = from_bits(oracle.gemm(bits(x), bits(w)))
    least = _lib.workspace_bytes(K.SK_OP_GEMM, M, N, Kd)
    ws_least = torch.zeros(max(least, 1), dtype=torch.uint8, device=DEV) if least else None
    assert_parity(K.gemm(xd, wd, ws=ws_least), ref, "least workspace")
    mm = K.SkinnyMatmul(M, N, Kd, DEV)
    out = mm(xd, wd)
    assert_parity(out, ref, "preferred workspace")
    # an explicit configuration on the same workspace, then the default plan again
    K.gemm(xd, wd, config=_lib.default_config(K.SK_OP_GEMM, M, N, Kd), ws=mm.ws)
    assert torch.equal(mm(xd, wd), out)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        mm(xd, wd)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = mm(xd, wd)
    for _ in range(3):
        captured.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, out)
        assert torch.equal(mm(xd, wd), out)


def test_stream_configs_are_planned():
    for N, Kd, cfg, ms in GEMM_CASES:
        for M in ms:
            assert _lib.check_config(K.SK_OP_GEMM, M, N, Kd, cfg) == SK_OK, (N, Kd, cfg, M)
    ok = lambda cfg, op=K.SK_OP_GEMM, M=16, N=6144, Kd=2560: _lib.check_config(op, M, N, Kd, cfg)
    assert ok(stream(24), M=17) == SK_ERR_CONFIG                  # one 16-row tile per K group
    assert ok(stream(24, 1, 2), M=65) == SK_OK                    # 64 rows, then one
    assert ok(stream(24, 1, 4, 4), M=129) == SK_OK                # 128 rows and one more launch
    assert ok(stream(96)) == SK_ERR_CONFIG                        # no six-slab instance
    assert ok(stream(24), Kd=2592) == SK_ERR_CONFIG               # K not whole units
    assert ok(stream(24, 41)) == SK_ERR_CONFIG                    # an empty split
    assert ok(stream(24), K.SK_OP_LM_ARGMAX) == SK_ERR_CONFIG
    assert ok(stream(40, 2), K.SK_OP_GATEUP, N=9728) == SK_ERR_CONFIG
    assert ok(stream(24), K.SK_OP_RESID_GEMM) == SK_ERR_CONFIG    # 24: not whole 16-column groups
    assert ok(stream(32), K.SK_OP_PRE_GEMM) == SK_ERR_CONFIG
    assert ok(tiles(256)) == SK_OK and ok(tiles(256), K.SK_OP_LM_ARGMAX) == SK_OK
    assert ok(tiles(256), Kd=2592) == SK_ERR_CONFIG
    for op in (K.SK_OP_GATEUP, K.SK_OP_RESID_GEMM, K.SK_OP_PRE_GEMM):   # logits and argmax only
        assert ok(tiles(256), op) == SK_ERR_CONFIG
    # counters (one per tile, padded to 256 bytes), then a block per tile and split
    assert _lib.workspace_bytes(K.SK_OP_GEMM, 16, 2560, 9728, stream(32, 3)) == 512 + 80 * 3 * 16 * 32 * 4
    assert _lib.workspace_bytes(K.SK_OP_GEMM, 5, 777, 2560, stream(10, 2)) == 512 + 78 * 2 * 5 * 12 * 4


def test_preferred_workspace_covers_the_least():
    for op, N, Kd in ((K.SK_OP_GEMM, 6144, 2560), (K.SK_OP_GEMM, 2560, 4096), (K.SK_OP_GEMM, 2560, 9728),
                      (K.SK_OP_GATEUP, 9728, 2560), (K.SK_OP_RMSNORM_GATEUP, 9728, 2560), (7, 2560, 9728),
                      (K.SK_OP_GEMM, 777, 2560), (K.SK_OP_LM_ARGMAX, 151936, 2560)):
        for M in (0, 1, 16, 17, 64, 65, 128):
            assert _lib.workspace_bytes_preferred(op, M, N, Kd) >= _lib.workspace_bytes(op, M, N, Kd), (op, N, M)
    assert _lib.workspace_bytes_preferred(K.SK_OP_GEMM, 16, 2560, 9728) == 512 + 80 * 3 * 16 * 32 * 4


@pytest.mark.gpu
@pytest.mark.parametrize("N,Kd,M", [(40960, 192, 130), (45001, 640, 177)])
def test_argmax_of_every_launch_of_a_call(N, Kd, M):
    """Past 128 rows the remainder is a launch of its own, with a plan of its
    own.  Bound: a logit is one bf16 rounding (half a unit of 8 significant
    bits, 2^-8 relative at most) away from the exact one, so the row's pick may
    trail the exact best by two."""
    g = torch.Generator().manual_seed(N + M)
    w, x = randn_bf16((N, Kd), 0.02, g).to(DEV), randn_bf16((M, Kd), 1.0, g).to(DEV)
    ids, maxv = K.LmArgmax(M, N, Kd, DEV)(x, w)
    exact = x.double() @ w.double().t()
    best = exact.max(-1).values
    picked = exact.gather(1, ids[:, None])[:, 0]
    step = 2.0 ** -8 * best * 1.01   # (fp32 accumulation: far below)
    assert bool((best - picked <= 2 * step).all())
    assert bool(((maxv.double() - picked).abs() <= step).all())


@pytest.mark.gpu
@pytest.mark.parametrize("N,Kd,grid,M", [(2577, 2048, 16, 100), (700, 4096, 44, 33), (3000, 320, 60, 64), (4100, 64, 256, 128),
                                         (1500, 2048, 9, 1)])
def test_stream_persistent_tiles_of_4_kb_strides(N, Kd, grid, M):
    """Row strides that are multiples of 4 KB: the workgroups start their tiles
    at units of their own, and a tile's first and last units wrap around."""
    g = torch.Generator().manual_seed(N + Kd + M)
    w, x = randn_bf16((N, Kd), 0.02, g), randn_bf16((M, Kd), 1.0, g)
    ld = (Kd + 2047) // 2048 * 2048
    wide = torch.full((N, ld), float("nan"), dtype=BF16, device=DEV)
    wide[:, :Kd] = w.to(DEV)
    xd, wd = x.to(DEV), wide[:, :Kd]
    out = K.gemm(xd, wd, config=tiles(grid))
    assert_parity(out, from_bits(oracle.gemm(bits(x), bits(w))), f"N={N} K={Kd} grid={grid} M={M}")
    ids, maxv = K.lm_argmax(xd, wd, config=tiles(grid))
    best = out.float().max(-1).values
    assert torch.equal(maxv, best) and torch.equal(ids, (out.float() == best[:, None]).float().argmax(-1))
