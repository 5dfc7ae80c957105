"""Prefill with the key ranges split over workgroups (a workspace given), against
the same call unsplit and, for sampled rows, against f64."""
import math

import pytest
import torch

from ullm_amd import _lib as L
from ullm_amd import attention as A

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _f64(q, k, v, rows, head, kvh, D, start, window):
    kk, vv = (t[:, kvh * D:(kvh + 1) * D].double().contiguous() for t in (k, v))
    s = q[rows, head * D:(head + 1) * D].double().contiguous() @ kk.t().contiguous() / math.sqrt(D)
    t = torch.arange(k.shape[0], device=q.device)[None]
    p = torch.tensor(rows, device=q.device)[:, None] + start
    hide = t > p
    if window:
        hide |= t <= p - window
    return torch.softmax(s.masked_fill(hide, -math.inf), -1) @ vv


# One row, rows on both sides of a unit (16, 32, 64, 128), ranges that end in
# and on a tile, GQA 1:1, 3:1, 4:1, 8:1, many parts (the merge's second batch),
# units with one part beside units with several, windows.
@pytest.mark.parametrize("dt,S,start,window,H,Hk,D", [
    ("bf16", 1, 4095, 0, 32, 8, 128), ("f16", 33, 3001, 0, 12, 4, 128), ("bf16", 129, 2000, 0, 32, 4, 128),
    ("f16", 8, 20000, 0, 8, 1, 128), ("bf16", 65, 4030, 0, 16, 16, 64), ("f16", 31, 6017, 0, 32, 8, 64),
    ("f32", 1, 4000, 0, 32, 8, 64), ("f32", 130, 3000, 0, 6, 2, 64), ("f32", 250, 300, 0, 6, 2, 64),
    ("f32", 40, 5000, 700, 32, 8, 64), ("f32", 17, 3333, 0, 32, 8, 128), ("f32", 100, 4000, 1500, 8, 8, 128),
    ("f16", 45, 5605, 0, 8, 4, 256), ("bf16", 5, 13493, 1024, 8, 4, 256), ("f32", 70, 2222, 0, 8, 4, 256),
    ("f32", 898, 0, 0, 12, 2, 128), ("f32", 217, 22, 1024, 8, 4, 256),
    # the longest unit a middle one: the first on the window's ramp, the last cut short
    ("f32", 1217, 0, 1024, 8, 4, 256), ("f32", 641, 1000, 1024, 8, 4, 256), ("f16", 1025, 4000, 4096, 8, 4, 256),
    ("bf16", 1621, 3000, 4096, 8, 4, 256), ("f16", 257, 1000, 1024, 8, 8, 256), ("f32", 1178, 0, 1024, 8, 8, 64),
    ("f32", 257, 1000, 1024, 32, 8, 64), ("f32", 257, 1000, 1024, 32, 8, 128),
])
@pytest.mark.parametrize("paged", [False, True])
def test_split_matches_unsplit_and_f64(dev, dt, S, start, window, H, Hk, D, paged):
    print(f"[prefill-split] {dt} S{S} start{start} win{window} {H}/{Hk}x{D} paged={paged}", flush=True)
    g = torch.Generator(device=dev).manual_seed(S + start)
    n = start + S
    q = torch.randn(S, H * D, device=dev, generator=g).to(DT[dt])
    k, v = (torch.randn(n, Hk * D, device=dev, generator=g).to(DT[dt]) for _ in range(2))
    if paged:
        P = 64
        pages = -(-n // P)
        order = torch.randperm(pages, generator=g, device=dev)
        kp, vp = (torch.zeros(pages, P, Hk * D, dtype=DT[dt], device=dev) for _ in range(2))
        for src, dst in ((k, kp), (v, vp)):
            padded = torch.zeros(pages * P, Hk * D, dtype=DT[dt], device=dev)
            padded[:n] = src
            dst[order] = padded.view(pages, P, -1)
        run = lambda: A.attn_prefill_paged(q, kp, vp, order.int(), H, Hk, D, start_pos=start, window=window)  # noqa: E731
    else:
        run = lambda: A.attn_prefill(q, k, v, H, Hk, D, start_pos=start, window=window)  # noqa: E731
    assert L.lib().ullm_hip_prefill_workspace_bytes(A._DT[DT[dt]], S, start, window, H, Hk, D) > 0
    split = run()
    whole = torch.empty_like(split)  # the entry points without a workspace
    if paged:
        L.check(L.lib().ullm_hip_attn_prefill_paged(
            A._ptr(q), A._ptr(kp), A._ptr(vp), A._DT[DT[dt]], Hk * D, 64, pages, A._ptr(order.int()), pages, S,
            start, window, H, Hk, D, 1 / math.sqrt(D), A._ptr(whole), A._stream()))
    else:
        L.check(L.lib().ullm_hip_attn_prefill(
            A._ptr(q), A._ptr(k), A._ptr(v), A._DT[DT[dt]], Hk * D, S, start, window, H, Hk, D,
            1 / math.sqrt(D), A._ptr(whole), A._stream()))
    # both hold P (and V of an f32 or bf16 cache) to f16's 2^-11
    assert float((split - whole).norm() / whole.norm()) <= 5e-4
    rows = sorted({0, S // 2, max(0, S - 40), S - 1})
    for h in (0, H - 1):
        ref = _f64(q, k, v, rows, h, h // (H // Hk), D, start, window)
        got = split[rows, h * D:(h + 1) * D].double()
        assert float((got - ref).norm() / ref.norm()) <= 1e-3


def test_small_workspace_runs_unsplit(dev):
    S, start, H, Hk, D = 9, 5000, 8, 2, 128
    print("[prefill-split] small workspace", flush=True)
    q = torch.randn(S, H * D, device=dev).to(torch.bfloat16)
    k, v = (torch.randn(start + S, Hk * D, device=dev).to(torch.bfloat16) for _ in range(2))
    n = L.lib().ullm_hip_prefill_workspace_bytes(L.DT_BF16, S, start, 0, H, Hk, D)
    outs = []
    for ws in (None, torch.empty(n - 1, dtype=torch.uint8, device=dev)):
        out = torch.empty(S, H * D, device=dev)
        L.check(L.lib().ullm_hip_attn_prefill_ws(
            A._ptr(q), A._ptr(k), A._ptr(v), L.DT_BF16, Hk * D, S, start, 0, H, Hk, D,
            1 / math.sqrt(D), A._ptr(out), A._ptr(ws), 0 if ws is None else n - 1, A._stream()))
        outs.append(out)
    assert torch.equal(*outs)


# Calls that are not split, with a window and a middle unit longer than the
# first and the last: a workspace given all the same is left alone.
@pytest.mark.parametrize("dt,S,start,window,H,Hk,D", [
    ("f32", 321, 16, 300, 32, 8, 64), ("f32", 385, 0, 129, 6, 2, 64),
    ("f32", 257, 0, 129, 6, 2, 128), ("f16", 257, 0, 129, 8, 8, 256), ("bf16", 300, 0, 100, 8, 2, 128),
])
def test_unsplit_call_leaves_workspace_alone(dev, dt, S, start, window, H, Hk, D):
    print(f"[prefill-unsplit-ws] {dt} S{S} start{start} win{window} {H}/{Hk}x{D}", flush=True)
    assert L.lib().ullm_hip_prefill_workspace_bytes(A._DT[DT[dt]], S, start, window, H, Hk, D) == 0
    g = torch.Generator(device=dev).manual_seed(S)
    q = torch.randn(S, H * D, device=dev, generator=g).to(DT[dt])
    k, v = (torch.randn(start + S, Hk * D, device=dev, generator=g).to(DT[dt]) for _ in range(2))
    ws = torch.full((8 << 20,), 0xA5, dtype=torch.uint8, device=dev)
    outs = []
    for w in (None, ws):
        out = torch.full((S, H * D), 7.0, device=dev)
        L.check(L.lib().ullm_hip_attn_prefill_ws(
            A._ptr(q), A._ptr(k), A._ptr(v), A._DT[DT[dt]], Hk * D, S, start, window, H, Hk, D,
            1 / math.sqrt(D), A._ptr(out), A._ptr(w), 0 if w is None else w.numel(), A._stream()))
        outs.append(out)
    assert torch.equal(*outs) and bool((ws == 0xA5).all())
    rows = list(range(0, S, 16)) + [S - 1]
    ref = _f64(q, k, v, rows, H - 1, Hk - 1, D, start, window)
    got = outs[1][rows, (H - 1) * D:].double()
    assert float((got - ref).norm() / ref.norm()) <= 1e-3


# The f32 head_dim-64 kernel unsplit: one set of waves (4 key tiles at most, or
# short windows on a full chip) and two, with 5 and odd tile counts, units whose
# second set has a tile less, and rows before the second set's keys.
@pytest.mark.parametrize("S,start,window,H,Hk", [(1, 0, 0, 8, 2), (127, 0, 0, 8, 8), (129, 0, 0, 4, 1), (161, 3, 0, 32, 8),
                                                 (777, 0, 0, 32, 8), (300, 0, 90, 6, 2), (2000, 0, 300, 32, 8)])
def test_f32_sets(dev, S, start, window, H, Hk):
    D = 64
    print(f"[prefill-f32-sets] S{S} start{start} win{window} {H}/{Hk}", flush=True)
    g = torch.Generator(device=dev).manual_seed(S)
    q = torch.randn(S, H * D, device=dev, generator=g)
    k, v = (torch.randn(start + S, Hk * D, device=dev, generator=g) for _ in range(2))
    out = torch.empty(S, H * D, device=dev)
    L.check(L.lib().ullm_hip_attn_prefill(A._ptr(q), A._ptr(k), A._ptr(v), L.DT_F32, Hk * D, S, start, window, H,
                                          Hk, D, 1 / math.sqrt(D), A._ptr(out), A._stream()))
    rows = list(range(0, S, max(1, S // 150))) + [S - 1]
    for h in (0, H - 1):
        ref = _f64(q, k, v, rows, h, h // (H // Hk), D, start, window)
        got = out[rows, h * D:(h + 1) * D].double()
        assert float((got - ref).norm() / ref.norm()) <= 1e-3
