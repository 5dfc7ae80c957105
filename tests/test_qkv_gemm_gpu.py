"""The many-row Q/K/V projection (ullm_hip_qkv_gemm_append): its GEMM against
an f64 product of the same inputs, its append against qkv_append, and the rule
that chooses it against the matvec path."""
import pytest
import torch

from tests.test_gemm_rule import MODES, SHAPES
from ullm_amd import attention as A

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _inputs(dev, rows, in_dim, H, Hk, D, wdt, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(rows, in_dim, device=dev, generator=g)
    ws = [(torch.randn(n * D, in_dim, device=dev, generator=g) / in_dim ** 0.5).to(DT[wdt])
          for n in (H, Hk, Hk)]
    return x, ws


def _raw(x, ws, H, Hk, D, bits, start=0):
    """The projections alone: no bias or norm, and a RoPE table of zero angles."""
    rows = x.shape[0]
    cs = torch.zeros(start + rows, D // 2, 2, device=x.device)
    cs[..., 0] = 1
    kc = torch.full((start + rows + 1, Hk * D), 7.0, device=x.device)
    vc = kc.clone()
    mv = None if bits else A.proj_workspace(rows, H, Hk, D, x.device)  # bits 0: the matvec per row
    q = A._F.proj(x, *ws, kc, vc, start, bits, cs, H, Hk, D, D, True, None, None, 1e-6, None, None, None,
                  None, None, None, mv, None)
    for c in (kc, vc):  # rows outside start.. are untouched
        assert bool((c[:start] == 7).all()) and bool((c[start + rows:] == 7).all())
    return q, kc[start:start + rows], vc[start:start + rows]


# Shapes that reach every tile, whole and split, with its edges (shown on the
# host: test_gemm_rule.py).
@pytest.mark.parametrize("wdt,bits", MODES)
@pytest.mark.parametrize("rows,in_dim,H,Hk,D", SHAPES)
def test_projection_vs_f64(dev, rows, in_dim, H, Hk, D, wdt, bits):
    print(f"[qkv-gemm] rows{rows} in{in_dim} H{H} Hk{Hk} D{D} {wdt} bits{bits}", flush=True)
    x, ws = _inputs(dev, rows, in_dim, H, Hk, D, wdt, 5)
    # rows over 2^-60 .. 2^60, the largest element 2^20 times the others in one
    x *= torch.exp2(torch.randint(-60, 61, (rows, 1), device=dev, dtype=torch.float32))
    x[0, 0] *= 2.0 ** 20
    # relative residual of the planes, plus the f32 additions (in_dim of them
    # at most); f16 planes also lose 2^-51 of the row's largest |x|
    eps = (2.0 ** -16 if bits == 16 else 2.0 ** -21) + in_dim * 2.0 ** -24
    for y, w in zip(_raw(x, ws, H, Hk, D, bits, start=2), ws):
        w64 = w.double()
        ref = x.double() @ w64.t().contiguous()
        bound = eps * (x.double().abs() @ w64.abs().t().contiguous())
        if wdt == "f16":
            bound += 2.0 ** -51 * x.double().abs().amax(1, keepdim=True) * w64.abs().sum(1)
        assert bool(((y.double() - ref).abs() <= bound + 1e-37).all())


@pytest.mark.parametrize("wdt", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("power,weight", [(0, 1), (5, 1), (10, 1), (20, 1), (10, 0), (15, 0), (20, 0)])
def test_error_is_no_larger_than_the_matvecs(dev, wdt, power, weight):
    """Against f64, also for rows with outliers, and where no weight takes the
    outliers (what is small beside them then is all of the result)."""
    rows, E, H, Hk, D = 64, 2048, 8, 4, 128
    print(f"[qkv-gemm-outlier] {wdt} 2^{power} weight {weight}", flush=True)
    x, ws = _inputs(dev, rows, E, H, Hk, D, wdt, 30 + power)
    for col in (7, 1203):
        x[:, col] *= 2.0 ** power
        for w in ws:
            w[:, col] *= weight
    ref = x.double() @ torch.cat(ws).double().t().contiguous()
    gemm, matvec = (float((torch.cat(_raw(x, ws, H, Hk, D, b), 1).double() - ref).norm() / ref.norm())
                    for b in (24, 0))
    print(f"gemm {gemm:.3g} matvec {matvec:.3g}", flush=True)
    assert gemm <= matvec


@pytest.mark.parametrize("wdt,bits", [("bf16", 16), ("bf16", 24), ("f16", 24), ("f32", 24)])
def test_infinities_and_nans_stay_in_their_rows(dev, wdt, bits):
    rows, in_dim, H, Hk, D = 40, 96, 2, 1, 64
    print(f"[qkv-gemm-inf] {wdt} bits{bits}", flush=True)
    x, ws = _inputs(dev, rows, in_dim, H, Hk, D, wdt, 6)
    clean = _raw(x, ws, H, Hk, D, bits)
    x2 = x.clone()
    x2[3, 5], x2[7, 0], x2[9, 90] = float("inf"), float("nan"), -3.4028e38
    x2[11] = 0
    got = _raw(x2, ws, H, Hk, D, bits)
    for y, c in zip(got, clean):
        keep = [r for r in range(rows) if r not in (3, 7, 9, 11)]
        assert torch.equal(y[keep], c[keep])
        assert bool((y[11] == 0).all())
    y, w = got[2], ws[2]  # v: no RoPE (whose zero sines make NaN of an infinity)
    assert torch.equal(y[3], torch.where(w[:, 5] > 0, float("inf"), -float("inf")))
    assert bool(torch.isnan(y[7]).all())
    ref = x2[9].double() @ w.double().t().contiguous()
    assert bool(((y[9].double() - ref).abs() <= 1e-4 * ref.abs()).all())


@pytest.mark.parametrize("wdt", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("rows,in_dim,H,Hk,D", [(40, 96, 2, 1, 64), (33, 2560, 4, 2, 128), (130, 1032, 4, 2, 128)])
def test_infinite_weights_stay_infinite(dev, wdt, rows, in_dim, H, Hk, D):
    """Infinities and NaNs among the weights give what f32 products and sums
    give, also for values of x with empty planes (1, 0)."""
    print(f"[qkv-gemm-winf] {wdt} rows{rows} in{in_dim}", flush=True)
    x, ws = _inputs(dev, rows, in_dim, H, Hk, D, wdt, 12)
    x[:, 7], x[2, 7], x[5, 90] = 1.0, 0.0, float("-inf")
    clean = _raw(x, ws, H, Hk, D, 24)
    inf = float("inf")
    for w in ws:
        w[5, 7], w[5, 11], w[9, in_dim - 1], w[11, 3], w[13, 90] = inf, inf, -inf, float("nan"), inf
    got, w = _raw(x, ws, H, Hk, D, 24)[2], ws[2]  # v: no RoPE (whose zero sines make NaN of an infinity)
    want = x.double() @ w.double().t().contiguous()
    odd = ~torch.isfinite(want)
    assert int(odd.sum()) > rows and bool(torch.isinf(want).any())
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)].float())
    keep = ~odd
    keep[:, [5, 9, 11, 13]] = False
    assert torch.equal(got[keep], clean[2][keep])


@pytest.mark.parametrize("kvdt", ["f32", "bf16"])
@pytest.mark.parametrize("rows,D,wdt,neox,rd", [(11, 256, "f16", True, 256), (50, 128, "bf16", False, 128),
                                                (70, 64, "f32", True, 32)])
def test_append_and_rule_match_matvec(dev, rows, D, wdt, neox, rd, kvdt, monkeypatch):
    """qkv_proj_append gives the same rows on both sides of its rule."""
    print(f"[qkv-gemm-append] rows{rows} D{D} {wdt} kv={kvdt}", flush=True)
    H, Hk, in_dim, start = 6, 2, 1536, 9
    x, ws = _inputs(dev, rows, in_dim, H, Hk, D, wdt, 8)
    cs = A.rope_table(start + rows, rd, 1e4, device=dev)
    g = torch.Generator(device=dev).manual_seed(9)
    qn, kn = (torch.randn(D, device=dev, generator=g) for _ in range(2))
    qb, kb, vb = (torch.randn(n * D, device=dev, generator=g) for n in (H, Hk, Hk))
    got = []
    for pays in (True, False):
        monkeypatch.setattr(A, "_gemm_pays", lambda *a: pays)
        kc = torch.zeros(start + rows, Hk * D, device=dev, dtype=DT[kvdt])
        vc = torch.zeros_like(kc)
        q = A.qkv_proj_append(x, *ws, kc, vc, cs, start_pos=start, n_head=H, n_kv_head=Hk, head_dim=D,
                              rotary_dim=rd, neox=neox, q_norm=qn, k_norm=kn, q_bias=qb, k_bias=kb,
                              v_bias=vb, q_dtype=DT[kvdt])
        got.append((q.float(), kc.float(), vc.float()))
    # f32 sums in another order; a 16-bit store can round one step (2^-7) apart
    for a, b in zip(*got):
        assert float((a - b).norm() / b.norm()) <= (2e-6 if kvdt == "f32" else 5e-4)
        step = 2.0 ** -7 * b.abs() if kvdt == "bf16" else 0
        assert bool(((a - b).abs() <= 2e-5 + step).all())


@pytest.mark.parametrize("rows", [2, 3, 5])
def test_few_row_prompts_share_no_counters(dev, rows, monkeypatch):
    """bf16 prompts of few rows: engines of one shape on two streams give what
    each gives alone, and none uses the process-wide projection workspace."""
    print(f"[few-rows] {rows}", flush=True)
    H, Hk, D, E = 32, 8, 128, 2560

    def no_cached(*a):
        raise AssertionError("the shared workspace")

    monkeypatch.setattr(A, "proj_workspace", no_cached)
    runs = []
    for i in range(2):
        ga = A.GpuAttention(A.AttnParams(1, H, Hk, D, 64, kv_dtype=torch.bfloat16))
        x, ws = _inputs(dev, rows, E, H, Hk, D, "bf16", 20 + i)
        runs.append((ga, x, ws, ga.forward_batch_proj(0, x, *ws, 0)))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in runs]
    outs = [[], []]
    for _ in range(20):
        for i, (ga, x, ws, _) in enumerate(runs):
            with torch.cuda.stream(streams[i]):
                outs[i].append(ga.forward_batch_proj(0, x, *ws, 0))
    torch.cuda.synchronize()
    for (_, _, _, want), got in zip(runs, outs):
        assert all(torch.equal(o, want) for o in got)
