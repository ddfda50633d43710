"""The plan that a call without a configuration takes (host logic of the library).

The stream path is chosen by shape and row range, and only where the workspace
holds its plan; the results of both sides are within the same bounds, so these
tests look at the choice itself, at both edges of every range.
"""

from __future__ import annotations

import pytest
import torch

from starter_amd import _lib
from starter_amd import kernels as K
from starter_amd._lib import SK_PATH_STREAM

GEMM, GATEUP, ARGMAX, RESID = K.SK_OP_GEMM, K.SK_OP_GATEUP, K.SK_OP_LM_ARGMAX, _lib.SK_OP_RESID_GEMM

# op, N, K, the row counts up to 128 that take the stream path
RANGES = [
    (GEMM, 6144, 2560, ((2, 128),)),
    (GEMM, 2560, 4096, ((17, 64), (97, 128))),
    (GEMM, 2560, 9728, ((3, 128),)),
    (GATEUP, 9728, 2560, ((17, 128),)),
    (RESID, 2560, 4096, ((17, 40), (49, 64), (97, 128))),
    (RESID, 2560, 9728, ((3, 128),)),
    (GEMM, 151936, 2560, ((33, 128),)),
    (ARGMAX, 151936, 2560, ((49, 128),)),
    (GEMM, 40960, 320, ((33, 128),)),
    (GEMM, 40959, 320, ()),            # fewer rows than a tile for every CU
    # beside a ring plan of seven waves and more: by the share of the tiles' rows that exist
    (GEMM, 41024, 2048, ()),           # 0.50
    (ARGMAX, 41024, 2048, ()),
    (GEMM, 41024, 1536, ((33, 128),)),     # six waves
    (GEMM, 41024, 2560, ((49, 128),)),     # ten waves, but two K splits past 48 rows
    (GEMM, 57344, 2048, ((49, 128),)),     # 0.70
    (ARGMAX, 57344, 2048, ((49, 128),)),
    (GEMM, 65536, 2048, ((41, 128),)),     # 0.80
    (GEMM, 81920, 2048, ((33, 128),)),     # 1.00
    (GEMM, 40960, 352, ()),            # K not whole 64-column units
    (GEMM, 777, 2560, ()),
]


@pytest.mark.parametrize("op,N,Kd,ranges", RANGES)
def test_stream_ranges(op, N, Kd, ranges):
    for M in range(1, 129):
        c = _lib.selected_config(op, M, N, Kd)
        inside = any(lo <= M <= hi for lo, hi in ranges)
        assert (c.path == SK_PATH_STREAM) == inside, (M, c)
        assert _lib.check_config(op, M, N, Kd, c) == _lib.SK_OK, (M, c)
        if not inside:
            assert c.as_dict() == _lib.default_config(op, M, N, Kd).as_dict(), M


@pytest.mark.parametrize("op,plain,N,Kd", [(_lib.SK_OP_RMSNORM_GEMM, GEMM, 6144, 2560),
                                           (_lib.SK_OP_RMSNORM_GATEUP, GATEUP, 9728, 2560),
                                           (_lib.SK_OP_RMSNORM_LM_ARGMAX, ARGMAX, 151936, 2560)])
def test_normed_calls_take_their_projections_plan(op, plain, N, Kd):
    for M in (2, 16, 17, 48, 49, 64, 65, 128):
        assert _lib.selected_config(op, M, N, Kd).as_dict() == _lib.selected_config(plain, M, N, Kd).as_dict(), M


def test_the_workspace_decides():
    """Down at 64 rows: four splits of 40-row tiles, three of 32 in the least
    workspace, and nothing in less."""
    N, Kd, M = 2560, 9728, 64
    least, most = _lib.workspace_bytes(GEMM, M, N, Kd), _lib.workspace_bytes_preferred(GEMM, M, N, Kd)
    assert least < most
    c = _lib.selected_config(GEMM, M, N, Kd, most)
    assert (c.path, c.rows, c.split) == (SK_PATH_STREAM, 40, 4)
    for n in (most - 1, least):
        c = _lib.selected_config(GEMM, M, N, Kd, n)
        assert (c.path, c.rows, c.split) == (SK_PATH_STREAM, 32, 3), n
    with pytest.raises(_lib.SkError) as e:
        _lib.selected_config(GEMM, M, N, Kd, least - 1)
    assert e.value.status == _lib.SK_ERR_WORKSPACE
    # at 16 rows the least workspace is none, and the table's plan runs in it
    assert _lib.workspace_bytes(GEMM, 16, N, Kd) == 0
    assert _lib.selected_config(GEMM, 16, N, Kd, 0).as_dict() == _lib.default_config(GEMM, 16, N, Kd).as_dict()


def test_pickers_log_the_plan_that_runs():
    """(The wrappers are built on the CPU here; only the plan is looked at.)"""
    lines = []
    K._log_choice(lines.append, "matmul", GEMM, 16, 2560, 9728)
    assert f"'path': {SK_PATH_STREAM}" in lines[0] and "'split': 3" in lines[0]
    a, w = torch.empty(64, 2560, dtype=K.BF16), torch.empty(6144, 2560, dtype=K.BF16)
    K.pick_matmul(a, w, lines.append)
    K.pick_normed("matmul", a[:1], a[:1], a[0], w, 1e-6, lines.append)
    assert f"'path': {SK_PATH_STREAM}" in lines[1] and "'path': 2" in lines[2]   # 1 row: the fused GEMV
