"""The choices of the many-row Q/K/V projection, on the host alone: the rule
that sends a call to the GEMM (attention._gemm_pays) against the measurements
that it rests on, and the tiles that the GEMM's tests reach."""
import ctypes as C

import pytest
import torch

from ullm_amd import _lib as L
from ullm_amd.attention import _gemm_pays

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16
MODES = [("bf16", 16), ("bf16", 24), ("f16", 24), ("f32", 24)]
# (rows, in_dim, n_head, n_kv_head, head_dim).  Rows on both sides of the token
# tiles (32, 64, 128), in_dim below a step, with a tail of 8, 24 and 40 dims, and
# long enough to be split over several ranges; from the ninth on each leaves part
# of the last token tile and of the last output tile (128, 256, 384) empty.
SHAPES = [
    (1, 8, 1, 1, 64), (31, 40, 3, 1, 64), (33, 264, 4, 2, 64), (64, 1048, 2, 2, 256),
    (65, 2560, 8, 4, 128), (129, 1032, 9, 3, 128), (383, 544, 32, 8, 64), (1025, 512, 16, 4, 128),
    (31, 1576, 31, 31, 64), (33, 40, 27, 9, 64), (33, 520, 27, 9, 64), (513, 40, 63, 21, 64),
    (150, 1032, 63, 21, 64), (33, 2600, 31, 31, 64), (333, 40, 31, 31, 64), (333, 520, 27, 9, 64),
    (650, 40, 31, 31, 64), (333, 1032, 31, 31, 64), (3000, 40, 27, 9, 64), (650, 1032, 31, 31, 64),
    (650, 520, 31, 31, 64),
]
DT = {"f32": L.DT_F32, "f16": L.DT_F16, "bf16": L.DT_BF16}


def plan(shape, wdt, bits):
    """(tokens of a tile, outputs of a tile, ranges of in_dim)"""
    p = (C.c_int32 * 3)()
    L.check(L.lib().ullm_hip_qkv_gemm_plan(shape[0], shape[1], DT[wdt], bits, *shape[2:], p))
    return tuple(p)


@pytest.mark.parametrize("wdt,bits", MODES)
def test_shapes_reach_every_tile_with_its_edges(wdt, bits):
    """Every tile of the mode, whole and in ranges of in_dim, at a shape that
    leaves part of its last token tile and of its last output tile empty."""
    seen = set()
    for shape in SHAPES:
        bs, bo, ks = plan(shape, wdt, bits)
        if shape[0] % bs and (shape[2] + 2 * shape[3]) * shape[4] % bo:
            seen.add((bs, bo, ks > 1))
    tiles = {(32, 256), (64, 128), (128, 128)}
    if wdt != "f32":
        tiles.add((64, 256))
    if bits == 16:
        tiles |= {(128, 256), (128, 384)}
    want = {(*t, s) for t in tiles for s in (False, True)}
    assert want <= seen, want - seen


def test_plan_validation():
    p = (C.c_int32 * 3)()
    f = L.lib().ullm_hip_qkv_gemm_plan
    assert f(16, 252, L.DT_F16, 24, 4, 2, 64, p) == L.E_UNSUPPORTED
    assert f(16, 256, L.DT_F16, 24, 4, 2, 64, None) == L.E_INVALID
    f = L.lib().ullm_hip_prefill_plan
    assert f(L.DT_F16, 16, 0, 0, 4, 2, 96, p) == L.E_UNSUPPORTED
    assert f(L.DT_F16, 16, 0, 0, 4, 2, 64, None) == L.E_INVALID


# (rows, outputs, in_dim, head_dim, weights): us as a matvec per row, as a GEMM
@pytest.mark.parametrize("call,matvec,gemm", [
    ((1, 18432, 16384, 128, BF16), 122, 152), ((1, 18432, 16384, 128, F16), 122, 170), ((2, 18432, 16384, 128, F16), 185, 171),
    ((2, 10240, 8192, 128, BF16), 62, 46), ((4, 6144, 2560, 128, BF16), 15, 20), ((12, 6144, 2560, 128, BF16), 29, 20),
    ((8, 3072, 2048, 64, F16), 10, 16), ((32, 3072, 2048, 64, F16), 27, 17),
    ((12, 6144, 2560, 128, F32), 56, 59), ((24, 6144, 2560, 128, F32), 86, 59), ((16, 6144, 4096, 128, F32), 86, 96),
    ((20, 6144, 4096, 128, F32), 109, 97), ((4, 10240, 8192, 128, F32), 137, 292), ((8, 10240, 8192, 128, F32), 235, 294),
    ((16, 10240, 8192, 128, F32), 369, 293), ((2, 18432, 16384, 128, F32), 365, 1165), ((8, 18432, 16384, 128, F32), 1070, 1183),
    ((12, 18432, 16384, 128, F32), 1529, 1176), ((8, 8192, 3584, 256, F32), 203, 91), ((6, 8192, 3584, 256, F32), 62, 91),
    ((2, 32768, 8192, 256, F32), 508, 912), ((4, 32768, 8192, 256, F32), 1005, 915), ((2, 32768, 8192, 256, BF16), 530, 116),
    ((1, 32768, 8192, 256, F16), 103, 123), ((8, 8192, 512, 256, F32), 27, 30),
    ((9, 8192, 512, 256, F32), 45, 30), ((8, 8192, 768, 256, F32), 39, 31), ((16, 4096, 2560, 256, BF16), 150, 20),
])
def test_rule_takes_the_faster_side(call, matvec, gemm):
    assert _gemm_pays(*call) == (gemm < matvec)
