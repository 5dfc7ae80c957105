"""The decode step with the append fused into the attention kernels
(GpuAttention.forward / forward_proj) against the append and the attention as
calls of their own."""
import pytest
import torch

from ullm_amd import _lib as L
from ullm_amd import attention as A

pytestmark = pytest.mark.gpu

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _engine(dev, kv, H, Hk, D, n_ctx, window, neox, seed):
    ga = A.GpuAttention(A.AttnParams(1, H, Hk, D, n_ctx, rope_theta=1e4, rope_neox=neox,
                                     sliding_window=window, kv_dtype=DT[kv]), device=dev)
    g = torch.Generator(device=dev).manual_seed(seed)
    for c in (ga.key_cache, ga.val_cache):
        c.copy_(torch.randn(c.shape, device=dev, generator=g))
    return ga, g


def _prep(dev, g, H, Hk, D, norm, bias):
    kw = {}
    if norm:
        kw.update(q_norm=torch.randn(D, device=dev, generator=g), k_norm=torch.randn(D, device=dev, generator=g))
    if bias:
        kw.update({n + "_bias": torch.randn(m * D, device=dev, generator=g) for n, m in (("q", H), ("k", Hk), ("v", Hk))})
    return kw


def _separate(ga, q, k, v, pos, kw):
    p = ga.p
    qr = A.qkv_append(q.view(1, -1), k.view(1, -1), v.view(1, -1), ga.key_cache[0], ga.val_cache[0], ga.rope_cs,
                      start_pos=pos, n_head=p.n_head, n_kv_head=p.n_kv_head, head_dim=p.head_dim,
                      neox=p.rope_neox, eps=p.eps, **kw)
    return A.attn_decode(qr.view(1, p.n_head, p.head_dim), ga.key_cache[0], ga.val_cache[0],
                         ga._lens[pos:pos + 1], pos + 1, p.n_kv_head, window=ga._window(0),
                         workspace=ga.workspace).view(-1)


# Positions on both sides of the fused range (33 old keys and more), of the 32-
# and 64-key splits and of the loop kernel, a window that binds, just binds and
# cannot; head_dim 256 and the first tokens take the separate launches.
@pytest.mark.parametrize("kv", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("pos,window,H,Hk,D,neox,norm,bias", [
    (0, 0, 8, 2, 64, True, True, False), (20, 0, 8, 2, 128, True, True, True), (32, 0, 8, 2, 64, False, False, True),
    (33, 0, 8, 2, 64, True, False, False), (64, 0, 32, 8, 64, False, True, True), (511, 0, 32, 8, 64, False, False, False),
    (2999, 0, 32, 8, 128, True, True, False), (4096, 0, 12, 2, 128, True, False, True), (700, 256, 8, 4, 128, True, True, True),
    (255, 256, 8, 4, 64, True, True, False), (256, 256, 8, 4, 64, False, True, False), (9000, 3000, 32, 4, 128, True, True, False),
    (20001, 0, 32, 4, 128, False, True, True), (33000, 0, 8, 8, 64, True, False, False), (1500, 0, 40, 2, 128, True, True, False),
    (1200, 0, 8, 4, 256, True, True, False),
])
def test_forward_matches_separate_calls(dev, kv, pos, window, H, Hk, D, neox, norm, bias):
    print(f"[token] kv={kv} pos{pos} win{window} {H}/{Hk}x{D} neox={neox} norm={norm} bias={bias}", flush=True)
    ga, g = _engine(dev, kv, H, Hk, D, pos + 2, window, neox, pos)
    kw = _prep(dev, g, H, Hk, D, norm, bias)
    q, k, v = (torch.randn(n * D, device=dev, generator=g) for n in (H, Hk, Hk))
    before = ga.key_cache.clone(), ga.val_cache.clone()
    out = ga.forward(0, q, k, v, pos, **kw)
    rows = [c[0, pos].float() for c in (ga.key_cache, ga.val_cache)]
    for c, b in zip((ga.key_cache, ga.val_cache), before):  # nothing but row pos changes
        c2 = c.clone()
        c2[0, pos] = b[0, pos]
        assert torch.equal(c2, b)
        c.copy_(b)
    ref = _separate(ga, q, k, v, pos, kw)
    # the same row up to the order of the norm's sum: one rounding step of its type
    step = {"f32": 2.0 ** -20, "f16": 2.0 ** -10, "bf16": 2.0 ** -7}[kv]
    for a, b in zip(rows, (ga.key_cache[0, pos].float(), ga.val_cache[0, pos].float())):
        assert bool(((a - b).abs() <= step * b.abs() + 1e-5).all())
    # P in f16 (f16 cache) or in hi + lo halves; the own key's in f32 here
    tol = {"f32": 2e-5, "f16": 5e-4, "bf16": 5e-4}[kv]
    assert float((out - ref).norm() / ref.norm()) <= tol


@pytest.mark.parametrize("w", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("pos,H,Hk,D,in_dim", [(40, 5, 1, 64, 8), (300, 12, 2, 128, 1544), (3000, 32, 8, 128, 2560),
                                               (600, 7, 7, 64, 520), (25, 8, 2, 128, 256)])
def test_forward_proj_matches_separate_calls(dev, w, pos, H, Hk, D, in_dim):
    print(f"[token-proj] w={w} pos{pos} {H}/{Hk}x{D} in{in_dim}", flush=True)
    ga, g = _engine(dev, "f32", H, Hk, D, pos + 1, 0, True, pos)
    kw = _prep(dev, g, H, Hk, D, True, True)
    x = torch.randn(in_dim, device=dev, generator=g)
    ws = [(torch.randn(n * D, in_dim, device=dev, generator=g) / in_dim ** 0.5).to(DT[w]) for n in (H, Hk, Hk)]
    out = ga.forward_proj(0, x, pos, *ws, **kw)
    raw = [(t.double() @ x.double()).float() for t in ws]
    ref = _separate(ga, *raw, pos, kw)
    assert float((out - ref).norm() / ref.norm()) <= 2e-5


def test_unaligned_rows_take_the_separate_launches(dev):
    H, Hk, D, pos = 8, 2, 64, 500
    ga, g = _engine(dev, "f16", H, Hk, D, pos + 1, 0, True, 3)
    buf = torch.randn((H + 2 * Hk) * D + 1, device=dev, generator=g)
    cut = [buf[1:][a:b] for a, b in ((0, H * D), (H * D, (H + Hk) * D), ((H + Hk) * D, (H + 2 * Hk) * D))]
    out = ga.forward(0, *cut, pos)
    assert torch.allclose(out, ga.forward(0, *[c.clone() for c in cut], pos), rtol=1e-3, atol=1e-4)


def test_graph_replays_match_eager(dev):
    H, Hk, D, pos = 32, 8, 64, 700
    ga, g = _engine(dev, "f16", H, Hk, D, pos + 1, 0, True, 5)
    q, k, v = (torch.randn(n * D, device=dev, generator=g) for n in (H, Hk, Hk))
    ga.forward(0, q, k, v, pos)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ga.forward(0, q, k, v, pos)
    for i in range(4):
        for t in (q, k, v):
            t.normal_(generator=g)
        want = ga.forward(0, q, k, v, pos).clone()
        ga.val_cache[0, pos] = 0
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), i


# An engine may project k and v straight into the slot of an f32 cache (a view
# as matmul's y): the append takes them in place, also with norms and biases.
@pytest.mark.parametrize("pos,window,H,Hk,D,neox", [(511, 0, 32, 8, 64, True), (2999, 0, 32, 4, 128, False),
                                                    (900, 256, 8, 4, 128, True)])
@pytest.mark.parametrize("which", ["kv", "k", "v"])
def test_rows_projected_into_the_cache(dev, pos, window, H, Hk, D, neox, which):
    print(f"[token-in-place] pos{pos} win{window} {H}/{Hk}x{D} {which}", flush=True)
    ga, g = _engine(dev, "f32", H, Hk, D, pos + 2, window, neox, pos)
    kw = _prep(dev, g, H, Hk, D, True, True)
    q, k, v = (torch.randn(n * D, device=dev, generator=g) for n in (H, Hk, Hk))
    before = ga.key_cache.clone(), ga.val_cache.clone()
    want = _separate(ga, q, k, v, pos, kw)
    rows = ga.key_cache.clone(), ga.val_cache.clone()
    for c, b, x, n in ((ga.key_cache, before[0], k, "k"), (ga.val_cache, before[1], v, "v")):
        c.copy_(b)
        if n in which:
            c[0, pos] = x
    got = ga.forward(0, q, ga.key_cache[0, pos] if "k" in which else k,
                     ga.val_cache[0, pos] if "v" in which else v, pos, **kw)
    assert torch.equal(got, want)
    assert torch.equal(ga.key_cache, rows[0]) and torch.equal(ga.val_cache, rows[1])
