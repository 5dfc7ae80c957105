"""Performance cases of the attention path: what an inference engine on top of
`ullm_amd.attention` has it do, over the range of sizes, types and options it
does it with.

A case is a dict of plain values.  `kind` names the call a program makes:

  decode       one decode step's attention over `layers` resident caches
               (attn_decode, the workspace kept by the caller)
  decode_step  one token through GpuAttention.forward, `layers` layers
               (bias/norm/RoPE + cache append, then attention)
  decode_proj  one token through GpuAttention.forward_proj, `layers` layers
               (Q/K/V projections with the append, then attention)
  paged_step   one token of every sequence of a ragged batch over paged caches
               (qkv_append_paged, attn_decode_paged)
  prefill      a prompt, or its next chunk, through GpuAttention.forward_batch
  prefill_paged  a chunk of a prompt over pages (attn_prefill_paged)
  block        a prompt, or its next chunk, from the normed hidden states
               through GpuAttention.forward_batch_proj

`prepare` makes the inputs on the GPU from the seed; `run` is one pass;
`exact` is the same result in 64-bit arithmetic, rounded only where the entry
points store a 16-bit value (the cache rows, and a prompt's q).
"""
import math

import torch

from ullm_amd import attention as A

DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}
EPS = 1e-6

# Attention shapes: n_head, n_kv_head, head_dim, hidden size, RoPE base,
# per-head Q/K norm, projection biases, NeoX pairing.
MODELS = {
    "llama-3.2-1b": (32, 8, 64, 2048, 5e5, False, False, False),
    "qwen2.5-1.5b": (12, 2, 128, 1536, 1e6, False, True, True),
    "qwen3-4b": (32, 8, 128, 2560, 1e6, True, False, True),
    "gemma-3-4b": (8, 4, 256, 2560, 1e6, True, False, True),
    "qwen3-30b-a3b": (32, 4, 128, 2048, 1e6, True, False, True),
}


def listed():
    return [
        # The smallest call: one layer of a small model in the reference's own
        # f32 cache, a short conversation.
        dict(name="decode_step_f32_512", kind="decode_step", model="llama-3.2-1b", kv="f32",
             len=512, window=0, layers=1),
        # A decode step's attention of a small model, 28 layers, 4K context.
        dict(name="decode_f16_4k", kind="decode", model="qwen2.5-1.5b", kv="f16", batch=1,
             len=4096, window=0, layers=28),
        # Long-context decode.
        dict(name="decode_bf16_32k", kind="decode", model="qwen3-30b-a3b", kv="bf16", batch=1,
             len=32768, window=0, layers=4),
        # A batched serving step: 8 sequences of different lengths over pages.
        dict(name="paged_step_b8", kind="paged_step", model="qwen3-30b-a3b", kv="bf16", batch=8,
             lo=4096, hi=32768, page=256),
        # One token from the hidden state, projections included.
        dict(name="decode_proj_bf16_3k", kind="decode_proj", model="qwen3-4b", kv="bf16",
             w="bf16", len=3001, window=0, layers=6),
        # A 2048-token prompt's attention.
        dict(name="prefill_bf16_2k", kind="prefill", model="qwen3-4b", kv="bf16", s=2048, start=0,
             window=0),
        # A sliding-window layer over a longer prompt of odd length.
        dict(name="prefill_f16_window_4k", kind="prefill", model="gemma-3-4b", kv="f16", s=4001,
             start=0, window=1024),
        # A prompt into the reference's f32 cache.
        dict(name="prefill_f32_777", kind="prefill", model="llama-3.2-1b", kv="f32", s=777,
             start=0, window=0),
        # Chunked prefill: 512 tokens that continue an 8K prompt, over pages.
        dict(name="prefill_paged_chunk", kind="prefill_paged", model="qwen3-4b", kv="bf16", s=512,
             start=7680, window=0, page=256),
        # A whole attention block of a 2048-token prompt, bf16 weights.
        dict(name="block_bf16_2k", kind="block", model="qwen3-4b", kv="bf16", w="bf16", s=2048,
             start=0, window=0),
        # The same block for a short chat turn that continues a conversation.
        dict(name="block_bf16_61", kind="block", model="qwen3-4b", kv="bf16", w="bf16", s=61,
             start=700, window=0),
        # A prompt through f16 weights and the f32 cache, as f16 model files
        # run.
        dict(name="block_f16_1k", kind="block", model="llama-3.2-1b", kv="f32", w="f16", s=1000,
             start=0, window=0),
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw(rng):
    kind = rng.choice(("decode", "decode_step", "decode_proj", "paged_step", "prefill",
                       "prefill_paged", "block", "block"))
    model = rng.choice(sorted(MODELS))
    kv = rng.choice(("f32", "f16", "bf16"))
    window = rng.choice((0, 1024)) if model == "gemma-3-4b" else 0
    c = dict(kind=kind, model=model, kv=kv)
    if kind == "decode":
        c.update(batch=rng.choice((1, 1, 2, 3, 4, 8)), len=_spread(rng, 64, 32768), window=window,
                 layers=_spread(rng, 1, 28))
    elif kind == "decode_step":
        c.update(len=_spread(rng, 64, 32768), window=window, layers=_spread(rng, 1, 16))
    elif kind == "decode_proj":
        c.update(w=rng.choice(("f32", "f16", "bf16")), len=_spread(rng, 64, 16384), window=window,
                 layers=_spread(rng, 1, 8))
    elif kind == "paged_step":
        hi = _spread(rng, 256, 32768)
        c.update(batch=_spread(rng, 2, 30), lo=max(1, hi // 8), hi=hi,
                 page=rng.choice((32, 64, 256)))
    else:
        s = _spread(rng, 2, 4096)
        start = rng.choice((0, 0, _spread(rng, 16, 16384)))
        c.update(s=s, start=start, window=window)
        if kind == "prefill_paged":
            c.update(page=rng.choice((64, 256)))
        if kind == "block":
            c.update(w=rng.choice(("bf16", "bf16", "f16", "f32")))
            if c["w"] != "bf16":
                c.update(s=_spread(rng, 2, 512))
    return c


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        c = _draw(rng)
        if _cost(c) <= most:
            return c


def _lengths(case):
    """A ragged batch's lengths, spread over [lo, hi] by its sizes alone."""
    b, lo, hi = case["batch"], case["lo"], case["hi"]
    return [lo + (i * 7919 * 31 + 12345) % (hi - lo + 1) for i in range(b)]


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, dtype=torch.float32, scale=1.0):
    x = torch.randn(*shape, device="cuda", generator=g)
    if scale != 1.0:
        x.mul_(scale)
    return x.to(dtype)


def _fill(g, t):
    """N(0, 1) values into a cache, a layer at a time."""
    for x in t:
        x.copy_(torch.randn(x.shape, device="cuda", generator=g))


def _params(g, case):
    """Norm weights and biases of a layer, for the models that have them."""
    H, Hk, D, _, _, norm, bias, _ = MODELS[case["model"]]
    kw = {}
    if norm:
        kw["q_norm"] = _randn(g, D, scale=0.2) + 1.0
        kw["k_norm"] = _randn(g, D, scale=0.2) + 1.0
    if bias:
        kw["q_bias"] = _randn(g, H * D, scale=0.5)
        kw["k_bias"] = _randn(g, Hk * D, scale=0.5)
        kw["v_bias"] = _randn(g, Hk * D, scale=0.5)
    return kw


def _engine(case, layers, n_ctx):
    H, Hk, D, _, theta, _, _, neox = MODELS[case["model"]]
    # One kind of layer per case: with a window the layers below the sixth
    # are sliding-window layers.
    return A.GpuAttention(A.AttnParams(
        n_layer=layers, n_head=H, n_kv_head=Hk, head_dim=D, n_ctx=n_ctx, rope_theta=theta,
        eps=EPS, rope_neox=neox, sliding_window=case["window"], kv_dtype=DT[case["kv"]]))


def _layer_ids(case):
    """`layers` layer numbers of the case's kind (every sixth is global)."""
    ids, l = [], 0
    while len(ids) < case["layers"]:
        if not (case["window"] and l % 6 == 5):
            ids.append(l)
        l += 1
    return ids


def prepare(case, seed):
    g = _gen(seed)
    H, Hk, D, E, theta, _, _, neox = MODELS[case["model"]]
    dt = DT[case["kv"]]
    kind = case["kind"]
    st = dict(case=case)
    if kind == "decode":
        B, L = case["batch"], case["len"]
        st["lens"] = torch.full((B,), L, dtype=torch.int32, device="cuda")
        st["ws"] = A.new_decode_workspace(B, H, Hk, D, L, case["window"])
        st["layers"] = [(_randn(g, B, H, D), _randn(g, B, L, Hk * D, dtype=dt),
                         _randn(g, B, L, Hk * D, dtype=dt)) for _ in range(case["layers"])]
    elif kind in ("decode_step", "decode_proj"):
        ids = _layer_ids(case)
        pos = case["len"] - 1
        ga = _engine(case, ids[-1] + 1, case["len"])
        _fill(g, ga.key_cache)
        _fill(g, ga.val_cache)
        layers = []
        for l in ids:
            kw = _params(g, case)
            if kind == "decode_step":
                ins = (_randn(g, H * D), _randn(g, Hk * D), _randn(g, Hk * D))
            else:
                ins = (_randn(g, E),)
                kw.update(_weights(g, case))
            layers.append((l, ins, kw))
        st.update(ga=ga, pos=pos, layers=layers)
    elif kind == "paged_step":
        lens, page = _lengths(case), case["page"]
        st.update(_pages(g, case, [n for n in lens]))
        st["lens"] = torch.tensor(lens, dtype=torch.int32, device="cuda")
        st["pos"] = st["lens"] - 1
        st["max_len"] = case["hi"]
        st["rope"] = A.rope_table(case["hi"], D, theta)
        B = case["batch"]
        st["q"], st["k"], st["v"] = (_randn(g, B, n * D) for n in (H, Hk, Hk))
        st["kw"] = _params(g, case)
        st["ws"] = torch.zeros(max(256, A.L.lib().ullm_hip_paged_decode_workspace_bytes(
            B, H, Hk, D, case["hi"], 0)), dtype=torch.uint8, device="cuda")
        # The slots that the step writes.
        at = [(st["pages_of"][b][(n - 1) // page], (n - 1) % page) for b, n in enumerate(lens)]
        st["new_k"] = [st["k_pages"][p, i] for p, i in at]
        st["new_v"] = [st["v_pages"][p, i] for p, i in at]
    elif kind == "prefill_paged":
        S, start = case["s"], case["start"]
        st.update(_pages(g, case, [start + S]))
        st["q"] = _randn(g, S, H * D, dtype=dt)
    else:
        S, start = case["s"], case["start"]
        ga = _engine(case, 1, start + S)
        _fill(g, ga.key_cache)
        _fill(g, ga.val_cache)
        kw = _params(g, case)
        if kind == "prefill":
            ins = tuple(_randn(g, S, n * D) for n in (H, Hk, Hk))
        else:
            ins = (_randn(g, S, E),)
            kw.update(_weights(g, case))
        st.update(ga=ga, ins=ins, kw=kw)
    return st


def _weights(g, case):
    H, Hk, D, E = MODELS[case["model"]][:4]
    return {n: _randn(g, m * D, E, dtype=DT[case["w"]], scale=1.0 / math.sqrt(E))
            for n, m in (("wq", H), ("wk", Hk), ("wv", Hk))}


def _pages(g, case, lens):
    """Pools of pages in shuffled order and the block table of the sequences."""
    Hk, D = MODELS[case["model"]][1:3]
    page, dt = case["page"], DT[case["kv"]]
    need = [-(-n // page) for n in lens]
    width = -(-max([case.get("hi", 0)] + lens) // page)
    order = torch.randperm(sum(need), generator=g, device="cuda").tolist()
    pages_of, at = [], 0
    for n in need:
        pages_of.append(order[at:at + n])
        at += n
    table = torch.tensor([p + [0] * (width - len(p)) for p in pages_of], dtype=torch.int32,
                         device="cuda")
    pools = [_randn(g, sum(need), page, Hk * D, dtype=dt) for _ in range(2)]
    return dict(k_pages=pools[0], v_pages=pools[1], table=table, pages_of=pages_of)


def run(st):
    case = st["case"]
    H, Hk, D = MODELS[case["model"]][:3]
    kind = case["kind"]
    if kind == "decode":
        L = case["len"]
        return [A.attn_decode(q, k, v, st["lens"], L, Hk, window=case["window"],
                              seq_stride=L * Hk * D, workspace=st["ws"])
                for q, k, v in st["layers"]]
    if kind in ("decode_step", "decode_proj"):
        ga, pos = st["ga"], st["pos"]
        outs = []
        for l, ins, kw in st["layers"]:
            if kind == "decode_step":
                o = ga.forward(l, *ins, pos, **kw)
            else:
                o = ga.forward_proj(l, *ins, pos, **kw)
            outs.append([o, ga.key_cache[l, pos], ga.val_cache[l, pos]])
        return outs
    if kind == "paged_step":
        q = A.qkv_append_paged(st["q"], st["k"], st["v"], st["k_pages"], st["v_pages"],
                               st["rope"], st["pos"], st["table"], n_head=H, n_kv_head=Hk,
                               head_dim=D, neox=MODELS[case["model"]][7], eps=EPS, **st["kw"])
        o = A.attn_decode_paged(q.view(-1, H, D), st["k_pages"], st["v_pages"], st["table"],
                                st["lens"], st["max_len"], Hk, workspace=st["ws"])
        return dict(out=o, k=st["new_k"], v=st["new_v"])
    if kind == "prefill_paged":
        return A.attn_prefill_paged(st["q"], st["k_pages"], st["v_pages"], st["table"][0], H, Hk,
                                    D, start_pos=case["start"], window=case["window"])
    ga, start, S = st["ga"], case["start"], case["s"]
    if kind == "prefill":
        o = ga.forward_batch(0, *st["ins"], start, **st["kw"])
    else:
        kw = dict(st["kw"])
        o = ga.forward_batch_proj(0, st["ins"][0], kw.pop("wq"), kw.pop("wk"), kw.pop("wv"),
                                  start, **kw)
    return dict(out=o, k=ga.key_cache[0, start:start + S], v=ga.val_cache[0, start:start + S])


def _pairs(s, start, window):
    """(query, key) pairs of a causal prompt chunk."""
    if not window:
        return s * start + s * (s + 1) // 2
    return sum(min(start + i + 1, window) for i in range(s))


def work(case):
    H, Hk, D, E = MODELS[case["model"]][:4]
    es = SIZE[case["kv"]]
    row = Hk * D * es  # bytes of one K or V cache row
    kind = case["kind"]
    win = case.get("window", 0)
    if kind in ("decode", "decode_step", "decode_proj"):
        keys = min(case["len"], win) if win else case["len"]
        seqs = case.get("batch", 1) * case["layers"]
        nbytes = seqs * (2 * keys * row + 8 * H * D)
        flops = seqs * 4 * keys * H * D
        if kind == "decode_step":
            nbytes += seqs * 4 * (H + 2 * Hk) * D
        if kind == "decode_proj":
            n = (H + 2 * Hk) * D * E
            nbytes += seqs * (n * SIZE[case["w"]] + 4 * E)
            flops += seqs * 2 * n
        return {"bytes": nbytes, "flops": flops}
    if kind == "paged_step":
        keys, b = sum(_lengths(case)), case["batch"]
        return {"bytes": 2 * keys * row + b * (8 * H * D + 8 * Hk * D),
                "flops": 4 * keys * H * D}
    S, start = case["s"], case["start"]
    keys = S + (min(start, win) if win else start)
    nbytes = 2 * keys * row + 4 * S * H * D
    flops = 4 * _pairs(S, start, win) * H * D
    if kind == "prefill_paged":
        nbytes += S * H * D * es
    elif kind == "prefill":
        nbytes += 4 * S * (H + 2 * Hk) * D
    else:
        n = (H + 2 * Hk) * D * E
        nbytes += 4 * S * E + n * SIZE[case["w"]]
        flops += 2 * S * n
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what the entry points differ from `exact` by.  Measured
    (relative 2-norm): a prompt 1.6e-4 to 2.6e-4 (P and V are f16 on the matrix
    cores); decode over an f16 cache 1.5e-4 (P in f16), over a bf16 or f32
    cache 3e-6 to 6e-6.  A stored 16-bit value can also fall on the other side
    of a rounding boundary: one bf16 step of a value is 2^-7 of it at most, and
    one such step in the shortest stored row (256 values) is up to 5e-4 of the
    row."""
    if case["kind"] in ("prefill", "prefill_paged", "block"):
        return {"rel": 1e-3, "max": 3e-2}
    if case["kv"] == "f32":
        return {"rel": 3e-5, "max": 1.2e-3}
    return {"rel": 1e-3, "max": 3e-2}


def _cos_sin(positions, D, theta):
    """(cos, sin) of the RoPE angles: the angles are defined in f32
    (1 / theta^(2i/D), times the position), their cos and sin are taken in
    64 bits."""
    i = torch.arange(0, D, 2, dtype=torch.float32)
    freq = torch.reciprocal(torch.pow(torch.tensor(theta, dtype=torch.float32), i / D))
    ang = (positions.to("cpu", torch.float32)[:, None] * freq[None, :]).double().cuda()
    return ang.cos(), ang.sin()


def _rope(x, cos, sin, neox):
    """x [rows, heads, D]; cos/sin [rows, D/2]."""
    c, s = cos[:, None, :], sin[:, None, :]
    if neox:
        a, b = x.chunk(2, -1)
        return torch.cat([a * c - b * s, a * s + b * c], -1)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)


def _append64(case, q, k, v, kw, positions):
    """bias, per-head norm and RoPE in 64 bits: q, k, v as [rows, heads, D]."""
    H, Hk, D, _, theta, _, _, neox = MODELS[case["model"]]
    cos, sin = _cos_sin(positions, D, theta)
    res = []
    for x, n, name in ((q, H, "q"), (k, Hk, "k"), (v, Hk, "v")):
        x = x.double().view(-1, n * D)
        if name + "_bias" in kw:
            x = x + kw[name + "_bias"].double()
        x = x.view(-1, n, D)
        if name != "v":
            if name + "_norm" in kw:
                x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * \
                    kw[name + "_norm"].double()
            x = _rope(x, cos, sin, neox)
        res.append(x)
    return res


def _stored(x, dt):
    """What a cache of this type holds of x."""
    return x.to(dt)


def _attend64(q, k, v, start, window):
    """q [S, H, D] at positions start.., k/v [T, Hk, D]: [S, H, D] in 64 bits."""
    S, H, D = q.shape
    Hk = k.shape[1]
    G = H // Hk
    out = torch.empty(S, H, D, dtype=torch.float64, device="cuda")
    step = max(1, (1 << 25) // k.shape[0])
    for j in range(Hk):
        kj, vj = k[:, j].double().t().contiguous(), v[:, j].double().contiguous()
        for r in range(0, S, step):
            n = min(step, S - r)
            pos = torch.arange(start + r, start + r + n, device="cuda")[:, None]
            t = torch.arange(k.shape[0], device="cuda")[None, :]
            hide = t > pos
            if window:
                hide |= t <= pos - window
            for h in range(j * G, j * G + G):
                sc = (q[r:r + n, h].double().contiguous() @ kj) / math.sqrt(D)
                sc.masked_fill_(hide, -math.inf)
                out[r:r + n, h] = torch.softmax(sc, -1) @ vj
    return out


def exact(case, seed):
    st = prepare(case, seed)
    H, Hk, D = MODELS[case["model"]][:3]
    kind, dt = case["kind"], DT[case["kv"]]
    if kind == "decode":
        L = case["len"]
        return [torch.cat([_attend64(q[b:b + 1], k[b].view(L, Hk, D), v[b].view(L, Hk, D), L - 1,
                                     case["window"]) for b in range(q.shape[0])])
                for q, k, v in st["layers"]]
    if kind in ("decode_step", "decode_proj"):
        ga, pos, outs = st["ga"], st["pos"], []
        positions = torch.tensor([pos])
        for l, ins, kw in st["layers"]:
            q, k, v = ins if kind == "decode_step" else _proj64(ins[0].view(1, -1), kw)
            q, k, v = _append64(case, q, k, v, kw, positions)
            kc, vc = ga.key_cache[l].view(-1, Hk, D), ga.val_cache[l].view(-1, Hk, D)
            kc[pos], vc[pos] = _stored(k[0], dt), _stored(v[0], dt)
            o = _attend64(q, kc[:pos + 1], vc[:pos + 1], pos, case["window"])
            outs.append([o.view(-1), k.reshape(-1), v.reshape(-1)])
        return outs
    if kind == "paged_step":
        lens, page = _lengths(case), case["page"]
        q, k, v = _append64(case, st["q"], st["k"], st["v"], st["kw"], st["pos"])
        out = []
        for b, n in enumerate(lens):
            st["new_k"][b].copy_(_stored(k[b].reshape(-1), dt))
            st["new_v"][b].copy_(_stored(v[b].reshape(-1), dt))
            kb, vb = (st[p][st["pages_of"][b]].view(-1, Hk, D)[:n]
                      for p in ("k_pages", "v_pages"))
            out.append(_attend64(q[b:b + 1], kb, vb, n - 1, 0))
        return dict(out=torch.cat(out), k=[x.reshape(-1) for x in k],
                    v=[x.reshape(-1) for x in v])
    S, start = case["s"], case["start"]
    if kind == "prefill_paged":
        kb, vb = (st[p][st["pages_of"][0]].view(-1, Hk, D)[:start + S]
                  for p in ("k_pages", "v_pages"))
        return _attend64(st["q"].view(S, H, D), kb, vb, start, case["window"]).view(S, H * D)
    ga, kw = st["ga"], st["kw"]
    q, k, v = st["ins"] if kind == "prefill" else _proj64(st["ins"][0], kw)
    q, k, v = _append64(case, q, k, v, kw, torch.arange(start, start + S))
    kc, vc = ga.key_cache[0].view(-1, Hk, D), ga.val_cache[0].view(-1, Hk, D)
    kc[start:start + S], vc[start:start + S] = _stored(k, dt), _stored(v, dt)
    o = _attend64(_stored(q, dt), kc[:start + S], vc[:start + S], start, case["window"])
    return dict(out=o.view(S, H * D), k=k.reshape(S, -1), v=v.reshape(S, -1))


def _proj64(x, kw):
    """The projections of the hidden states, in 64 bits."""
    x = x.double()
    return tuple(x @ kw[n].double().t().contiguous() for n in ("wq", "wk", "wv"))
