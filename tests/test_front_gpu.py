"""The native front end of attention.py: errors, returned tensors, layer
indices, and calls on a stream that is not torch's current one."""
import pytest
import torch

from ullm_amd import _lib as L
from ullm_amd import attention as A

pytestmark = pytest.mark.gpu

H, Hk, D, N = 8, 2, 64, 300
NL = 5000  # keys enough for a prefill of 9 rows to be split, with scratch


def _cache(dev, dtype=torch.float16, n=N):
    g = torch.Generator(device=dev).manual_seed(4)
    k, v = (torch.randn(n, Hk * D, device=dev, generator=g).to(dtype) for _ in range(2))
    return torch.randn(1, H, D, device=dev, generator=g), k, v, torch.tensor([n], dtype=torch.int32, device=dev)


@pytest.mark.parametrize("change,code", [
    (dict(q=lambda q: q.cpu()), L.E_INVALID), (dict(q=lambda q: q.half()), L.E_INVALID),
    (dict(q=lambda q: q.transpose(1, 2)), L.E_INVALID), (dict(lens=lambda t: t.long()), L.E_INVALID),
    (dict(k=lambda k: k.double()), L.E_UNSUPPORTED), (dict(ws=lambda _: torch.empty(8, dtype=torch.uint8, device="cuda")), L.E_WORKSPACE),
])
def test_errors_keep_their_codes(dev, change, code):
    q, k, v, lens = _cache(dev)
    a = dict(q=q, k=k, v=v, lens=lens, ws=None)
    for n, f in change.items():
        a[n] = f(a[n])
    with pytest.raises(L.UllmHipError) as e:
        A.attn_decode(a["q"], a["k"], a["v"], a["lens"], N, Hk, workspace=a["ws"])
    assert e.value.code == code
    with pytest.raises(TypeError):
        A.attn_decode(q, None, v, lens, N, Hk)


def test_given_out_is_returned_and_written(dev):
    q, k, v, lens = _cache(dev)
    out = torch.full((1, H, D), 7.0, device=dev)
    assert A.attn_decode(q, k, v, lens, N, Hk, out=out) is out
    assert torch.equal(out, A.attn_decode(q, k, v, lens, N, Hk))


def test_other_stream_owns_its_scratch(dev):
    """Scratch of calls queued on another stream is not handed out while they
    wait there: the calls give what they give on the current stream."""
    q, k, v, lens = _cache(dev, n=NL)
    qp = torch.randn(9, H * D, device=dev).half()
    want = A.attn_decode(q, k, v, lens, NL, Hk), A.attn_prefill(qp, k, v, H, Hk, D, start_pos=NL - 9)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        torch.cuda._sleep(20_000_000)
    outs = [torch.empty_like(w) for w in want]
    A.attn_decode(q, k, v, lens, NL, Hk, out=outs[0], stream=s)
    A.attn_prefill(qp, k, v, H, Hk, D, start_pos=NL - 9, out=outs[1], stream=s)
    for _ in range(8):  # would take the scratch if it were free
        torch.full((1 << 20,), 0xFF, dtype=torch.uint8, device=dev)
        torch.full((256,), 0xFF, dtype=torch.uint8, device=dev)
    s.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(outs, want))


def test_scratch_comes_from_the_given_streams_memory(dev, monkeypatch):
    """A block that work queued on torch's current stream may still write is not
    handed to a call on another stream: its scratch is that stream's own."""
    q, k, v, lens = _cache(dev, n=NL)
    qp = torch.randn(9, H * D, device=dev).half()
    x, ws = torch.randn(64, 2048, device=dev), [torch.randn(n * D, 2048, device=dev).half() for n in (H, Hk, Hk)]
    cs = A.rope_table(64, D, 1e4, device=dev)
    monkeypatch.setattr(A, "_gemm_pays", lambda *a: True)
    assert L.lib().ullm_hip_prefill_workspace_bytes(L.DT_F16, 9, NL - 9, 0, H, Hk, D) > 0
    calls = [lambda s: A.attn_decode(q, k, v, lens, NL, Hk, out=torch.empty_like(q), stream=s),
             lambda s: A.attn_prefill(qp, k, v, H, Hk, D, start_pos=NL - 9, out=torch.empty(9, H * D, device=dev), stream=s),
             lambda s: A.qkv_proj_append(x, *ws, k, v, cs, start_pos=0, n_head=H, n_kv_head=Hk, head_dim=D, stream=s)]
    for i, call in enumerate(calls):
        s = torch.cuda.Stream()
        torch.cuda.synchronize()
        call(s)
        torch.cuda.synchronize()
        assert [b for b in torch.cuda.memory_snapshot() if b["stream"] == s.cuda_stream], \
            f"call {i}: its scratch came from another stream's memory"
        assert torch.cuda.current_stream().cuda_stream != s.cuda_stream


def test_calls_do_without_scratch_they_cannot_have(dev, monkeypatch):
    """With memory for the outputs alone, the split prefill runs unsplit and the
    projection of many rows row by row, as both did before they had scratch."""
    S, start, E, rows = 64, 60000, 2048, 1500
    k, v = (torch.randn(start + S, Hk * D, device=dev).half() for _ in range(2))
    q, out = torch.randn(S, H * D, device=dev).half(), torch.empty(S, H * D, device=dev)
    x, ws = torch.randn(rows, E, device=dev), [torch.randn(n * D, E, device=dev).half() / 45 for n in (H, Hk, Hk)]
    cs = A.rope_table(rows, D, 1e4, device=dev)
    kc, vc, qo = (torch.empty(rows, n * D, device=dev) for n in (Hk, Hk, H))
    kw = dict(start_pos=0, n_head=H, n_kv_head=Hk, head_dim=D)
    monkeypatch.setattr(A, "_gemm_pays", lambda *a: True)
    lib = L.lib()
    need = min(lib.ullm_hip_prefill_workspace_bytes(L.DT_F16, S, start, 0, H, Hk, D),
               lib.ullm_hip_qkv_gemm_workspace_bytes(rows, E, L.DT_F16, 24, H, Hk, D))
    assert need > 4 << 20  # more than a small-block segment of the allocator holds
    whole = torch.empty_like(out)
    L.check(lib.ullm_hip_attn_prefill(A._ptr(q), A._ptr(k), A._ptr(v), L.DT_F16, Hk * D, S, start, 0, H, Hk, D,
                                      D ** -0.5, A._ptr(whole), A._stream()))
    monkeypatch.setattr(A, "_gemm_pays", lambda *a: False)
    want = A.qkv_proj_append(x, *ws, kc.clone(), vc.clone(), cs, **kw)
    monkeypatch.setattr(A, "_gemm_pays", lambda *a: True)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / torch.cuda.mem_get_info()[1])
    try:
        pad = []
        with pytest.raises(torch.OutOfMemoryError):  # the allocator's free blocks
            while len(pad) < 1024:
                pad.append(torch.empty(2 << 20, dtype=torch.uint8, device=dev))
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(need, dtype=torch.uint8, device=dev)
        A.attn_prefill(q, k, v, H, Hk, D, start_pos=start, out=out)
        A.qkv_proj_append(x, *ws, kc, vc, cs, q_out=qo, **kw)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(out, whole) and torch.equal(qo, want)


@pytest.mark.parametrize("window", [-1, N, 2 ** 31 - 1, 2 ** 31, 2 ** 63 - 1])
def test_windows_that_hide_nothing(dev, window):
    q, k, v, lens = _cache(dev)
    qp = torch.randn(9, H * D, device=dev).half()
    assert torch.equal(A.attn_decode(q, k, v, lens, N, Hk, window=window), A.attn_decode(q, k, v, lens, N, Hk))
    assert torch.equal(A.attn_prefill(qp, k, v, H, Hk, D, start_pos=N - 9, window=window),
                       A.attn_prefill(qp, k, v, H, Hk, D, start_pos=N - 9))
    outs = []
    for w in (0, window):
        ga = A.GpuAttention(A.AttnParams(1, H, Hk, D, N, sliding_window=w))
        ga.key_cache[0], ga.val_cache[0] = k, v
        outs.append(ga.forward(0, q.view(-1), torch.ones(Hk * D, device=dev), torch.ones(Hk * D, device=dev), 200))
    assert torch.equal(*outs)


def test_calls_with_scratch_replay_from_a_graph(dev):
    """Few-row and GEMM projections, a split prefill and the decode step
    (fused, and with rows in the cache), captured together: each replay on new
    inputs, with eager work between, gives what the calls give eagerly."""
    H, Hk, D, E, n = 32, 8, 128, 2560, 4200
    gen = torch.Generator(device=dev).manual_seed(8)
    rn = lambda *s: torch.randn(*s, device=dev, generator=gen)  # noqa: E731
    ga, gf = (A.GpuAttention(A.AttnParams(1, H, Hk, D, n, kv_dtype=t)) for t in (torch.bfloat16, torch.float32))
    w = [(rn(m * D, E) / 50).bfloat16() for m in (H, Hk, Hk)]
    x3, x70, q, kv = rn(3, E), rn(70, E), rn(H * D), rn(2, Hk * D)

    def step():
        gf.key_cache[0, 4100], gf.val_cache[0, 4100] = kv[0], kv[1]
        return [ga.forward_batch_proj(0, x3, *w, 4000), ga.forward_batch_proj(0, x70, *w, 4010),
                ga.forward(0, q, kv[0], kv[1], 4090), gf.forward(0, q, kv[0], kv[1], 4099),
                gf.forward(0, q, gf.key_cache[0, 4100], gf.val_cache[0, 4100], 4100)]

    step()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = step()
    for _ in range(4):
        for t in (x3, x70, q, kv):
            t.copy_(rn(*t.shape))
        want = [o.clone() for o in step()]
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(outs, want))


def test_layer_indices(dev):
    ga = A.GpuAttention(A.AttnParams(3, H, Hk, D, 16, kv_dtype=torch.float32))
    q, kk = torch.randn(H * D, device=dev), torch.randn(Hk * D, device=dev)
    ga.forward(-1, q, kk, kk, 5)
    assert bool(ga.key_cache[2, 5].any()) and not bool(ga.key_cache[:2].any())
    for bad in (3, -4):
        with pytest.raises(IndexError):
            ga.forward(bad, q, kk, kk, 5)
