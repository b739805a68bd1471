"""Performance cases of the int8 paged KV cache: the calls a serving program makes,
at the shapes of the models the benchmark and the tests use.

A case names a `kind` of call, the attention shape (Hq query heads, Hkv KV heads,
head_dim D), the batch B, the context lengths U[lo, hi] and the options:

* decode    one decode step: RoPE optional, the new token's K/V appended and every query
            attended over its sequence's whole cache (fused call; `graph`: the step of all
            `layers` replayed from a HIP graph, as a serving loop runs it)
* chunk     `new` rows per sequence (speculative drafts, a prefill chunk, a whole prompt):
            quantize-append, then causal attention of those rows over the cache
* wdecode   the decode step of a sliding-window layer
* wchunk    a prefill chunk of a sliding-window layer
* cascade   a decode step of sequences forked from one shared prefix
* roundtrip prompts appended, their int8 snapshot taken, restored into fresh blocks and
            read back dequantized (prefix store and restore)
"""
import math

import numpy as np
import torch

import krill_amd
from krill_amd import _lib as KL
from krill_amd.pool import rope_table

BF16, F16, F32 = "bf16", "f16", "f32"
_TORCH = {BF16: torch.bfloat16, F16: torch.float16, F32: torch.float32}

# attention shapes of the models that the benchmark names
LLAMA_1B = dict(Hq=32, Hkv=8, D=64)
LLAMA_8B = dict(Hq=32, Hkv=8, D=128)
QWEN_14B = dict(Hq=40, Hkv=8, D=128)
QWEN_30B = dict(Hq=32, Hkv=4, D=128)
GEMMA3 = dict(Hq=16, Hkv=8, D=256)
GEMMA4 = dict(Hq=16, Hkv=2, D=512)

_DEFAULT = dict(B=1, lo=1, hi=1, new=1, layers=1, graph=False, rope=False, quant="affine_g64", dt=BF16, out=BF16,
                window=0, prefix=0, outliers=False)


def _case(kind, shape, **kw):
    c = dict(kind=kind, **shape, **_DEFAULT)
    c.update(kw)
    return c


def listed():
    return [
        # one user's chat on a small model: latency and launches, all layers of a step
        _case("decode", LLAMA_1B, name="step_b1", B=1, lo=2048, hi=2048, layers=16, graph=True, rope=True),
        # a serving batch at mixed contexts: the benchmark's headline layer
        _case("decode", QWEN_14B, name="decode_b32", B=32, lo=512, hi=8192),
        # few very long contexts, K with outlier channels
        _case("decode", QWEN_30B, name="decode_128k", B=8, lo=98304, hi=131072, outliers=True),
        # full-attention layers with head_dim 512, default output type
        _case("decode", GEMMA4, name="decode_head512", B=32, lo=512, hi=8192, out=F32),
        # speculative decoding: 8 drafted rows per sequence verified
        _case("chunk", LLAMA_8B, name="verify_k8", B=16, lo=1024, hi=8192, new=8),
        # chunked prefill of a batch on top of its contexts, K rotated in the append
        _case("chunk", QWEN_14B, name="prefill_chunk", B=8, lo=2048, hi=6144, new=512, rope=True),
        # a whole prompt from scratch in the reference's own row storage, fp16 model
        _case("chunk", LLAMA_8B, name="prefill_rows", B=1, lo=0, hi=0, new=3900, quant="ref_row", dt=F16, out=F16),
        # prefill of head_dim 512 layers
        _case("chunk", GEMMA4, name="prefill_head512", B=2, lo=700, hi=3000, new=256),
        # sliding-window layers: decode and prefill
        _case("wdecode", GEMMA3, name="window_decode", B=32, lo=512, hi=8192, window=1024, rope=True),
        _case("wchunk", GEMMA3, name="window_prefill", B=4, lo=300, hi=5000, new=512, window=1024),
        # many conversations behind one system prompt
        _case("cascade", LLAMA_8B, name="shared_prefix", B=64, lo=0, hi=1024, prefix=4096 + 24),
        # prefix entries written and restored
        _case("roundtrip", LLAMA_8B, name="prefix_roundtrip", B=4, lo=1500, hi=4096, rope=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "chunk", "chunk", "chunk", "wdecode", "wchunk", "cascade", "roundtrip"])
    quant = rng.choice(["affine_g64", "affine_g64", "ref_row"])
    dt = rng.choice([BF16, BF16, F16])
    out = rng.choice([dt, F32])
    common = dict(quant=quant, dt=dt, out=out)
    if kind == "decode":
        shape = rng.choice([LLAMA_1B, LLAMA_8B, QWEN_14B, QWEN_30B, GEMMA3, GEMMA4])
        B = _log(rng, 1, 64)
        hi = _log(rng, 64, min(131072, (1 << 18) // B))
        return _case(kind, shape, B=B, lo=max(1, hi // rng.choice([1, 2, 16])), hi=hi, rope=rng.random() < 0.5, **common)
    if kind == "chunk":
        shape = rng.choice([LLAMA_1B, LLAMA_8B, QWEN_14B, QWEN_30B, GEMMA3, GEMMA4])
        new = _log(rng, 2, 2000 if shape["D"] <= 256 else 200)
        most = 8 if shape["D"] <= 256 else 2
        B = max(1, min(16, _log(rng, 1, 16), most * 256 // new))
        hi = _log(rng, 1, 6000 if shape["D"] <= 256 else 3000)
        return _case(kind, shape, B=B, lo=hi // rng.choice([1, 2, 16]), hi=hi, new=new, rope=rng.random() < 0.5, **common)
    if kind in ("wdecode", "wchunk"):
        shape = rng.choice([GEMMA3, GEMMA3, LLAMA_8B])
        hi = _log(rng, 64, 8192)
        window = rng.choice([512, 1024, 1024, 2048])
        if kind == "wdecode":
            return _case(kind, shape, B=_log(rng, 1, 48), lo=max(1, hi // rng.choice([1, 4])), hi=hi, window=window,
                         rope=rng.random() < 0.7, **common)
        new = _log(rng, 16, 700)
        return _case(kind, shape, B=max(1, min(8, 2048 // new)), lo=hi // 4, hi=hi, new=new, window=window, **common)
    if kind == "cascade":
        shape = rng.choice([LLAMA_8B, QWEN_14B, LLAMA_1B])
        return _case(kind, shape, B=_log(rng, 4, 64), lo=0, hi=_log(rng, 16, 1500), prefix=_log(rng, 200, 6000), **common)
    shape = rng.choice([LLAMA_1B, LLAMA_8B, QWEN_30B, GEMMA3])
    hi = _log(rng, 40, 4096)
    return _case(kind, shape, B=_log(rng, 1, 6), lo=max(1, hi // 3), hi=hi, rope=rng.random() < 0.5, **common)


# ------------------------------------------------------------------ inputs


def _rng(seed, *what):
    return np.random.default_rng([int(seed) & 0x7FFFFFFF, *what])


def _lens(c, seed):
    """Context lengths before the call's new rows.  Their mean is held near the range's
    middle, so that one seed's work is another's."""
    if c["hi"] == c["lo"]:
        return [c["hi"]] * c["B"]
    u = (np.arange(c["B"]) + _rng(seed, 1).random(c["B"])) / c["B"]
    if c["B"] == 1:
        u = u * 0.1 + 0.45
    return [int(x) for x in _rng(seed, 2).permutation(np.floor(c["lo"] + u * (c["hi"] - c["lo"] + 1)).astype(np.int64))]


def _mean_len(c):
    return 0.5 * (c["lo"] + c["hi"])


def _gen(seed, *what):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(_rng(seed, 7, *what).integers(1 << 62)))
    return g


def _randn(c, seed, shape, *what):
    """N(0, 1) in the case's input type."""
    return torch.randn(shape, generator=_gen(seed, *what), device="cuda", dtype=torch.float32).to(_TORCH[c["dt"]])


def _kv(c, seed, b, T, layer=0):
    """K and V [1, Hkv, T, D] of sequence b (b = -1: the shared prefix); with outliers, 1 % of
    the K channels x20."""
    shape = (1, c["Hkv"], T, c["D"])
    k, v = _randn(c, seed, shape, 11, b + 1, layer), _randn(c, seed, shape, 12, b + 1, layer)
    if c["outliers"]:
        ch = _rng(seed, 3).choice(c["D"], size=max(1, c["D"] // 100), replace=False)
        k[..., torch.from_numpy(ch).cuda()] *= 20.0
    return k, v


def _scale(c):
    return 1.0 if c["D"] == 512 else 1.0 / math.sqrt(c["D"])


def _q(c, seed, layer=0):
    shape = (c["B"], c["Hq"], c["new"], c["D"])
    q = _randn(c, seed, shape, 13, layer)
    return q * 0.044 if c["D"] == 512 else q  # normed queries of the scale-1.0 layers


def _i32(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()


def _table(max_pos, D):
    return torch.from_numpy(rope_table(max_pos, D)).cuda()


def _pool(c, blocks, layers=1):
    return krill_amd.KVPool(layers, c["Hkv"], c["D"], blocks, c["quant"], c["dt"], free_list_seed=5)


def _append(pool, layer, k, v, slots):
    pool.quantize_append(layer, k.contiguous(), v.contiguous(), _i32(np.asarray(slots).reshape(1, -1)))


def _fill(c, seed, pool, lens, layers=1, window=False):
    """Sequences of `lens` tokens; a windowed pool keeps its last tokens only, so those
    are appended in chunks."""
    seqs = []
    for b, T in enumerate(lens):
        s = pool.seq_create()
        seqs.append(s)
        step = 512 if window else max(T, 1)
        kv = [_kv(c, seed, b, T, layer) for layer in range(layers)] if T else []
        for t in range(0, T, step):
            n = min(step, T - t)
            slots = pool.reserve_append(s, n).copy()
            for layer in range(layers):
                _append(pool, layer, kv[layer][0][:, :, t:t + n], kv[layer][1][:, :, t:t + n], slots)
    return seqs


def _blocks(lens, more):
    return sum((n + more + 63) // 64 + 1 for n in lens) + 8


def prepare(c, seed):
    lens, B, new = _lens(c, seed), c["B"], c["new"]
    st = dict(case=c, scale=_scale(c), out_dtype=_TORCH[c["out"]])
    kind = c["kind"]
    if kind == "roundtrip":
        return _prepare_roundtrip(c, seed, lens, st)
    if kind == "cascade":
        return _prepare_cascade(c, seed, lens, st)
    L = c["layers"]
    window = c["window"]
    pool = _pool(c, _blocks(lens, new), L)
    if window:
        pool.set_option(KL.OPT_WINDOW, window)
    seqs = _fill(c, seed, pool, lens, L, bool(window))
    slots = np.stack([pool.reserve_append(s, new).copy() for s in seqs])
    mx = max(lens) + new
    mb = (mx + 63) // 64
    tables, n = pool.batch_tables(seqs, mb)
    st.update(pool=pool, mx=mx, tables=_i32(tables), lens=_i32(n), slots=_i32(slots), window=window)
    if window:
        st["starts"] = _i32(pool.batch_starts(seqs))
    kv = [_new_kv(c, seed, layer) for layer in range(L)]
    st["k"], st["v"] = [x[0] for x in kv], [x[1] for x in kv]
    st["q"] = [_q(c, seed, layer) for layer in range(L)]
    st["o"] = torch.empty((L, B, c["Hq"], new, c["D"]), dtype=st["out_dtype"], device="cuda")
    if c["rope"]:
        st["cs"] = _table(mx + 64, c["D"])
        st["pos"] = _i32(np.asarray(lens)[:, None] + np.arange(new)[None, :])
    if window:
        need = _window_ws(pool, B, c["Hq"], new, mb, mx, window)
    else:
        need = pool.workspace_size(B, c["Hq"], new, mx)
    st["ws"] = torch.empty(max(need, 1), dtype=torch.uint8, device="cuda")
    if c["graph"]:
        _decode(st)
        torch.cuda.synchronize()
        g, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        with torch.cuda.graph(g, stream=side):
            _decode(st)
        torch.cuda.synchronize()
        st["replay"] = g
    return st


def _new_kv(c, seed, layer=0):
    shape = (c["B"], c["Hkv"], c["new"], c["D"])
    return _randn(c, seed, shape, 21, layer), _randn(c, seed, shape, 22, layer)


def _window_ws(pool, B, Hq, Lq, mb, mx, window):
    import ctypes

    need = ctypes.c_size_t()
    KL.check(KL.lib().krill_window_workspace_size(pool.handle, B, Hq, Lq, mb, mx, window, ctypes.byref(need)))
    return need.value


def _prepare_cascade(c, seed, lens, st):
    P, B = c["prefix"], c["B"]
    pool = _pool(c, (P + 63) // 64 + _blocks(lens, P % 64 + 1) + B)
    root = pool.seq_create()
    k, v = _kv(c, seed, -1, P)
    _append(pool, 0, k, v, pool.reserve_append(root, P).copy())
    seqs = [pool.seq_fork(root, P) for _ in range(B)]
    for b, T in enumerate(lens):
        if T:
            k, v = _kv(c, seed, b, T)
            _append(pool, 0, k, v, pool.reserve_append(seqs[b], T).copy())
    for s in seqs:
        pool.reserve_append(s, 1)
    pool.flush()
    pb = P // 64
    mb = (P + max(lens) + 1 + 63) // 64
    tables, n = pool.batch_tables(seqs, mb)
    sfx = np.asarray(n) - 64 * pb
    k, v = _new_kv(c, seed)
    st.update(pool=pool, prefix_table=_i32(tables[0, :pb]), tables=_i32(tables[:, pb:]), lens=_i32(sfx), mx=int(sfx.max()),
              q=_q(c, seed), k=k, v=v,
              o=torch.empty((B, c["Hq"], 1, c["D"]), dtype=st["out_dtype"], device="cuda"))
    st["ws"] = torch.empty(max(1, pool.shared_prefix_workspace_size(B, c["Hq"], pb, st["mx"])), dtype=torch.uint8, device="cuda")
    return st


def _prepare_roundtrip(c, seed, lens, st):
    B, S = c["B"], c["hi"]  # rows of the snapshots: the longest a prompt may be
    pool = _pool(c, 2 * _blocks(lens, 0))
    k = torch.zeros((B, c["Hkv"], S, c["D"]), dtype=_TORCH[c["dt"]], device="cuda")
    v = torch.zeros_like(k)
    slots, fresh = np.full((B, S), -1, np.int32), np.full((B, S), -1, np.int32)
    first, second = [], []
    for b, T in enumerate(lens):
        k[b:b + 1, :, :T], v[b:b + 1, :, :T] = _kv(c, seed, b, T)
        first.append(pool.seq_create())
        second.append(pool.seq_create())
        slots[b, :T] = pool.reserve_append(first[b], T)
        fresh[b, :T] = pool.reserve_append(second[b], T)
    mb = (S + 63) // 64
    t1, n = pool.batch_tables(first, mb)
    t2, _ = pool.batch_tables(second, mb)
    st.update(pool=pool, k=k, v=v, slots=_i32(slots), fresh=_i32(fresh), tables=_i32(t1), tables2=_i32(t2), lens=_i32(n), S=S,
              src=_i32(np.zeros(B)))
    if c["rope"]:
        st["cs"] = _table(S, c["D"])
        st["pos"] = _i32(np.broadcast_to(np.arange(S), (B, S)))
    return st


# --------------------------------------------------------------------- run


def _decode(st):
    p = st["pool"]
    for layer in range(st["case"]["layers"]):
        args = (layer, st["q"][layer], st["k"][layer], st["v"][layer], st["tables"], st["lens"], st["mx"], st["scale"])
        kw = dict(out_dtype=st["out_dtype"], ws=st["ws"], out=st["o"][layer])
        if st["case"]["rope"]:
            p.decode_append_attention_rope(*args, st["cs"], **kw)
        else:
            p.decode_append_attention(*args, **kw)
    return st["o"]


def run(st):
    c, p = st["case"], st["pool"]
    kind = c["kind"]
    if kind == "decode":
        if c["graph"]:
            st["replay"].replay()
            return st["o"]
        return _decode(st)
    if kind == "cascade":
        return p.attention_shared_prefix(0, st["q"], st["prefix_table"], st["tables"], st["lens"], st["mx"], st["scale"],
                                         out_dtype=st["out_dtype"], ws=st["ws"], out=st["o"], k_new=st["k"], v_new=st["v"])
    if kind == "roundtrip":
        if c["rope"]:
            p.quantize_append_rope(0, st["k"], st["v"], st["slots"], st["pos"], st["cs"])
        else:
            p.quantize_append(0, st["k"], st["v"], st["slots"])
        snap = p.gather(0, st["tables"], st["lens"], st["S"])
        p.scatter(0, snap, st["src"], st["fresh"])
        k, v = p.gather_dequant(0, st["tables2"], st["lens"], st["S"])
        return {"k": k, "v": v, "snap": snap}
    q, k, v, o = st["q"][0], st["k"][0], st["v"][0], st["o"][0]
    if kind == "wdecode":
        return p.decode_append_attention_windowed(0, q, k, v, st["tables"], st["lens"], st["starts"], st["window"], st["mx"],
                                                  st["scale"], cos_sin=st.get("cs"), out_dtype=st["out_dtype"],
                                                  ws=st["ws"], out=o)
    if c["rope"]:
        p.quantize_append_rope(0, k, v, st["slots"], st["pos"], st["cs"])
    else:
        p.quantize_append(0, k, v, st["slots"])
    if kind == "wchunk":
        return p.attention_windowed(0, q, st["tables"], st["lens"], st["starts"], st["window"], st["mx"], st["scale"],
                                    out_dtype=st["out_dtype"], ws=st["ws"], out=o)
    return p.attention(0, q, st["tables"], st["lens"], st["mx"], st["scale"], st["out_dtype"], ws=st["ws"], out=o)


def _size(t):
    return {BF16: 2, F16: 2, F32: 4}[t]


def work(c):
    """Bytes: the cached keys and values that the new rows see, once per KV head, the new rows in
    and out of the quantizer, queries and outputs.  Operations: two products per seen (row, key)."""
    B, Hq, Hkv, D, new, L = (c[k] for k in ("B", "Hq", "Hkv", "D", "new", "layers"))
    G = D // 64 if c["quant"] == "affine_g64" else 1
    tok = 2 * Hkv * D + 8 * Hkv * G  # one cached token of a layer
    row = 2 * Hkv * D * 2            # its K and V in the input type
    mean = _mean_len(c)
    if c["kind"] == "roundtrip":
        used, out = B * mean, B * c["hi"]
        return {"bytes": used * (row + 3 * tok) + out * (2 * tok + 2 * Hkv * D * 2), "flops": 0}
    if c["kind"] == "cascade":
        keys = c["prefix"] + B * (mean + 1)
        seen = B * (c["prefix"] + mean + 1)
    else:
        end = mean + new
        w = c["window"]
        if w and mean > 0:
            keys = B * min(end, w + new - 1)
            seen = B * new * min(mean + 0.5 * (new + 1), w)
        else:
            keys = B * end
            seen = B * new * (mean + 0.5 * (new + 1))
    qo = B * Hq * new * D * (2 + _size(c["out"]))
    return {"bytes": L * (keys * tok + B * new * (row + tok) + qo), "flops": L * 4 * Hq * D * seen}


def tolerance(c):
    """bf16 and fp16 outputs: their rounding, 2^-9 and 2^-12 of each value at the root mean
    square 1.7e-3 and 2.1e-4 from the 64-bit result.  fp32 outputs: a softmax and sums in fp32."""
    if c["kind"] == "roundtrip":
        return {"rel": 1e-3, "max": 2e-3}
    rel = {BF16: 7e-3, F16: 9e-4, F32: 2e-5}[c["out"]]
    return {"rel": rel, "max": 8 * rel}


# ------------------------------------------------- the same in 64 bits


def _div(a, b):
    """float32 quotient, rounded once (the 64-bit quotient rounded to 32 bits)."""
    return (a.double() / b.double()).float()


def _quantized(c, x):
    """The values the cache holds for rows x [..., D] in the input type, in 64 bits: the
    storage's bytes are defined by these 32-bit steps."""
    if c["quant"] == "affine_g64":
        w = x.half().float().unflatten(-1, (-1, 64))
        lo, hi = w.amin(-1, keepdim=True), w.amax(-1, keepdim=True)
        side = lo.abs() > hi.abs()
        s = _div(hi - lo, torch.full_like(lo, 255.0)).clamp_min(1e-7)
        s = torch.where(side, s, -s)
        edge = torch.where(side, lo, hi)
        q0 = torch.round(_div(edge, s))
        some = q0 != 0
        s = torch.where(some, _div(edge, torch.where(some, q0, torch.ones_like(q0))), s)
        bias = torch.where(some, edge, torch.zeros_like(edge))
        q = torch.round(_div(w - bias, s)).clamp(0, 255)
        return (q.double() * s.half().double() + bias.half().double()).flatten(-2)
    f = x.float()
    lo, hi = f.amin(-1, keepdim=True), f.amax(-1, keepdim=True)
    safe = _div((hi - lo).to(x.dtype).float(), torch.full_like(lo, 255.0)).clamp_min(1e-8)
    q = torch.trunc(_div((f - lo).to(x.dtype).float(), safe).clamp(0, 255))
    # the reference dequantizes with two fp16 roundings
    return ((q.double() * safe.half().double()).half().double() + lo.half().double()).half().double()


def _rotated(c, x, pos):
    """x [..., n, D] turned by positions pos [n], in 32 bits, rounded to the input type."""
    h = c["D"] // 2
    cs = torch.from_numpy(rope_reference(int(pos.max()) + 1, c["D"])).cuda()[pos]
    co, si = cs[:, :h], cs[:, h:]
    a, b = x[..., :h].float(), x[..., h:].float()
    return torch.cat([a * co - b * si, a * si + b * co], -1).to(x.dtype)


def rope_reference(max_pos, D, base=10000.0):
    ang = np.arange(max_pos, dtype=np.float64)[:, None] * base ** (-2.0 * np.arange(D // 2) / D)[None, :]
    return np.concatenate([np.cos(ang), np.sin(ang)], axis=1).astype(np.float32)


def _attend(c, q, k, v, first, window):
    """q [Hq, n, D] at positions first .. first + n - 1 over k, v [Hkv, T, D] (64 bits)."""
    R = c["Hq"] // c["Hkv"]
    n, T = q.shape[1], k.shape[1]
    p = torch.arange(n, device="cuda")[:, None] + first
    t = torch.arange(T, device="cuda")[None, :]
    hide = t > p
    if window:
        hide = hide | (t < p - window + 1)
    out = torch.empty_like(q)
    for h in range(c["Hkv"]):
        s = (q[h * R:(h + 1) * R].reshape(R * n, -1) @ k[h].T) * _scale(c)
        s = s.view(R, n, T).masked_fill(hide, -math.inf)
        w = torch.softmax(s, -1).view(R * n, T)
        out[h * R:(h + 1) * R] = (w @ v[h]).view(R, n, -1)
    return out


def exact(c, seed):
    lens = _lens(c, seed)
    if c["kind"] == "roundtrip":
        shape = (c["B"], c["Hkv"], c["hi"], c["D"])
        k = torch.zeros(shape, dtype=torch.float64, device="cuda")
        v = torch.zeros_like(k)
        for b, T in enumerate(lens):
            kb, vb = _kv(c, seed, b, T)
            if c["rope"]:
                kb = _rotated(c, kb, torch.arange(T, device="cuda"))
            k[b, :, :T], v[b, :, :T] = _quantized(c, kb)[0], _quantized(c, vb)[0]
        return {"k": k, "v": v, "snap": None}
    out = []
    for layer in range(c["layers"]):
        q = _q(c, seed, layer)
        kn, vn = _new_kv(c, seed, layer)
        rows = []
        for b, T in enumerate(lens):
            old = [_kv(c, seed, b, T, layer)] if T else []
            if c["prefix"]:
                old = [_kv(c, seed, -1, c["prefix"])] + old
                T += c["prefix"]
            pos = torch.arange(T, T + c["new"], device="cuda")
            kb, qb = kn[b:b + 1], q[b]
            if c["rope"]:
                kb = _rotated(c, kb, pos)
                if c["kind"] in ("decode", "wdecode"):
                    qb = _rotated(c, qb, pos)
            keys = torch.cat([_quantized(c, x[0][0]) for x in old] + [_quantized(c, kb[0])], 1)
            values = torch.cat([_quantized(c, x[1][0]) for x in old] + [_quantized(c, vn[b])], 1)
            rows.append(_attend(c, qb.double(), keys, values, T, c["window"]))
        out.append(torch.stack(rows))
    return torch.stack(out) if c["kind"] == "decode" else out[0]
