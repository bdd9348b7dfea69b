"""CPU: which instance of the many-row int8 launch a shape takes, and that the GPU test's shapes reach
every instance (test_gpu_int8_rows.py compares them with float64)."""

from __future__ import annotations

import pytest

from runtime_amd.phase2 import _hip
from test_gpu_int8_rows import GATEUP, LINEAR

INSTANCES = {(rows, npw) for rows in (2, 4, 6, 8) for npw in (2, 4)}  # (16-row tiles, n-tiles per wave)


def _plan(m: int, n: int, k: int, gateup: bool):
    v = _hip.load().mx_w8a16_rows_plan(m, n, k, int(gateup))
    return (v & 255, v >> 8 & 255, v >> 16) if v else None


@pytest.mark.parametrize("gateup", [False, True])
def test_gpu_shapes_reach_every_instance(gateup):
    shapes = [(m, 2 * n if gateup else n, k) for m, n, k, _ in (GATEUP if gateup else LINEAR)]
    plans = [(s, _plan(*s, gateup)) for s in shapes]
    plans = [(s, p) for s, p in plans if p]
    assert {p[:2] for _, p in plans} == INSTANCES
    for inst in INSTANCES:
        mine = [s for s, p in plans if p[:2] == inst]
        assert any(m % (16 * inst[0]) for m, _, _ in mine), f"{inst}: no shape with rows left over"
        assert any(n // 16 % (4 * inst[1]) for _, n, _ in mine), f"{inst}: no shape with channels left over"
    # The loop of two stages (8, 4) at odd and even k-tile counts; the loops of 3 (the other wide
    # ones) and 12 (the narrow ones) at several remainders.
    assert {k // 64 % 2 for (_, _, k), p in plans if p[:2] == (8, 4)} == {0, 1}
    assert {k // 64 % 3 for (_, _, k), p in plans if p[1] == 4 and p[0] < 8} == {0, 1, 2}
    assert len({k // 64 % 12 for (_, _, k), p in plans if p[1] == 2 and p[2] == 1}) >= 4
    assert gateup or {p[2] for _, p in plans if p[1] == 2} >= {1, 4}


def test_rows_that_stay_with_the_decode_launches():
    assert _plan(128, 4096, 4096, False) is None and _plan(129, 4096, 4096, False)
    assert _plan(64, 28672, 4096, True) is None and _plan(65, 28672, 4096, True)
    assert _plan(300, 4100, 4096, False) is None and _plan(300, 4096, 100, False) is None  # not whole tiles
