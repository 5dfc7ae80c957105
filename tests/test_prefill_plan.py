"""The split of prefill key ranges over workgroups (ullm_hip_prefill_plan), on
the host alone: no unit of any call may need more parts than are launched and
have scratch, whichever of its units is the longest."""
import ctypes as C

import numpy as np
import pytest

from ullm_amd import _lib as L

SHAPES = [(L.DT_F32, 8, 4, 256), (L.DT_F16, 8, 4, 256), (L.DT_BF16, 8, 8, 256), (L.DT_F32, 32, 8, 128),
          (L.DT_F32, 6, 2, 128), (L.DT_F32, 32, 8, 64), (L.DT_F32, 8, 8, 64), (L.DT_F32, 6, 2, 64),
          (L.DT_F16, 12, 2, 128), (L.DT_BF16, 6, 2, 64)]
STARTS = (0, 5, 300, 1000, 1016, 3000, 4000, 9000)


def unit_tiles(rows, tile, S, start, window):
    """Key tiles of every unit, from the header's description."""
    u = np.arange(-(-S // rows))
    lo = np.maximum(start + u * rows + 1 - window, 0) if window > 0 else 0 * u
    hi = start + np.minimum((u + 1) * rows, S)
    return -(-hi // tile) - lo // tile


def plan(dt, S, start, window, H, Hk, D):
    p = (C.c_int32 * 4)()
    L.check(L.lib().ullm_hip_prefill_plan(dt, S, start, window, H, Hk, D, p))
    return tuple(p)


def check(dt, S, start, window, H, Hk, D):
    """The call's parts, after its plan is seen to hold for every unit."""
    rows, tile, chunk, parts = plan(dt, S, start, window, H, Hk, D)
    longest = int(unit_tiles(rows, tile, S, start, window).max())
    assert -(-longest // chunk) <= parts, (dt, S, start, window, H, Hk, D, chunk, parts, longest)
    assert parts > 1 or chunk >= 1 << 26  # unsplit: no unit of any length is cut (2^31 keys are 2^26 tiles)
    need = parts * S * H * (D * 4 + 8) if parts > 1 else 0  # O and (m, l) planes of every part
    assert L.lib().ullm_hip_prefill_workspace_bytes(dt, S, start, window, H, Hk, D) == need
    return parts


@pytest.mark.parametrize("window", [0, 33, 128, 300, 700, 1024, 2048, 4096])
@pytest.mark.parametrize("dt,H,Hk,D", SHAPES)
def test_no_unit_needs_more_parts_than_planned(dt, H, Hk, D, window):
    lengths = sorted({*range(2, 300, 7), *range(301, 4200, 29), 257, 641, 853, 1016, 1025, 1178, 1217, 1248, 1621, 2113})
    for start in STARTS:
        for S in lengths:
            check(dt, S, start, window, H, Hk, D)


# A first unit still on the window's ramp and a last one cut short, so that a
# middle unit is the longest; all of them are split.
RAMPED = [(L.DT_F32, 1217, 0, 1024, 8, 4, 256), (L.DT_F32, 641, 1000, 1024, 8, 4, 256),
          (L.DT_F32, 853, 300, 1024, 8, 4, 256), (L.DT_F16, 1025, 4000, 4096, 8, 4, 256),
          (L.DT_BF16, 1621, 3000, 4096, 8, 4, 256), (L.DT_F16, 257, 1000, 1024, 8, 8, 256),
          (L.DT_F32, 1178, 0, 1024, 8, 8, 64), (L.DT_F32, 257, 1000, 1024, 32, 8, 64),
          (L.DT_F32, 257, 1000, 1024, 32, 8, 128)]


@pytest.mark.parametrize("case", RAMPED)
def test_ramped_first_and_short_last_unit(case):
    assert check(*case) > 1
