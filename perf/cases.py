"""The workloads that the attention library is timed on: one layer call each, as a serving program makes it.

A case is a dict of plain values:
  kind      which public entry point(s) run: see run()
  kv, io    storage type of the KV cache, and of Q and O: "f16", "bf16" or "fp32"
  B, T      sequences, and query tokens per sequence
  NQ, NKV, HD   query heads, KV heads, head dim
  lo, hi    context lengths (keys before the query tokens) are drawn uniformly from [lo, hi], from `lens`
  lens      seed of the lengths and of the draft trees (they belong to the case: its work depends on them)
  window    sliding window in keys (0: plain causal)
  chunk     split chunk given to the decode / verify entry points (0: the library's own)
  split     key split given to the prefill entry point (0: none, -1: chosen by the library)

Shapes are those of this repository's configurations: 24 q-heads over 4 KV heads of 256 (Qwen3.5 full attention),
16 over 8 of 256 (Gemma4 sliding layers), 16 over 1 of 512 (Gemma4 global layers), 16 over 4 of 128.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dgx-serving_amd"))
import dgx_attn as A  # noqa: E402

DT = {"fp32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"fp32": 4, "f16": 2, "bf16": 2}


def _case(kind, kv, io, B, T, NQ, NKV, HD, lo, hi, name=None, lens=1, window=0, chunk=0, split=0):
    c = dict(kind=kind, kv=kv, io=io, B=B, T=T, NQ=NQ, NKV=NKV, HD=HD, lo=lo, hi=hi, lens=lens, window=window,
             chunk=chunk, split=split)
    return dict(c, name=name) if name else c


def listed():
    return [
        # One user, one token, a short context, through the drop-in launcher: latency and launches.
        _case("decode_split", "f16", "fp32", 1, 1, 16, 4, 128, 511, 511, name="decode_one"),
        # A full serving batch: ragged contexts up to 8K, one token per sequence (the headline decode).
        _case("batch", "f16", "f16", 16, 1, 24, 4, 256, 255, 8191, name="decode_batch", lens=2026, chunk=512),
        # A sliding-window layer's decode step with its producers: norm + RoPE of q and k, norm of v, the cache
        # append and the windowed attention.
        _case("layer", "bf16", "bf16", 8, 1, 16, 8, 256, 1023, 4095, name="decode_layer_window", lens=9, window=1024,
              chunk=96),
        # A global layer's decode over long contexts: one KV head of 512.
        _case("batch", "bf16", "bf16", 8, 1, 16, 1, 512, 1023, 32767, name="decode_global", lens=13, chunk=512),
        # fp32 caches (the models that force them), ragged batch, through the drop-in launcher.
        _case("decode_f32", "fp32", "fp32", 16, 1, 24, 4, 256, 255, 8191, name="decode_fp32", lens=2026),
        # Speculative decoding: 8-node draft trees of 16 sequences verified in one call.
        _case("tree", "f16", "f16", 16, 8, 24, 4, 256, 2048, 16384, name="tree_verify", lens=5, chunk=640),
        # One user's 7-token draft verified through the drop-in launcher.
        _case("flash", "bf16", "fp32", 1, 7, 24, 4, 256, 3001, 3001, name="verify_one"),
        # A prompt of 1024 tokens (the headline prefill).
        _case("prefill", "bf16", "bf16", 1, 1024, 16, 8, 256, 0, 0, name="prefill_causal"),
        # A prompt of odd length with six q-heads per KV head, fp32 Q and O, through the drop-in launcher.
        _case("flash_v2", "f16", "fp32", 1, 1377, 24, 4, 256, 0, 0, name="prefill_gqa6"),
        # A prompt chunk over a cached prefix.
        _case("prefill", "bf16", "bf16", 1, 512, 16, 8, 256, 4096, 4096, name="prefill_chunked", split=-1),
        # A long prompt through a sliding-window layer.
        _case("prefill", "bf16", "bf16", 1, 4096, 16, 8, 256, 0, 0, name="prefill_window", window=1024),
        # A prompt through a global layer: one KV head of 512.
        _case("prefill", "bf16", "bf16", 1, 1024, 16, 1, 512, 0, 0, name="prefill_global"),
    ]


def draw(rng):
    def size(lo, hi):                      # spread over the logarithm
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    def short(kv, io, B, T, heads, hi, **kw):
        top = size(max(64, hi // 64), hi)
        return (kv, io, B, T) + heads, dict(lo=max(16, top // 8), hi=top, lens=rng.randrange(1 << 20), **kw)

    q35, slide, glob, small = (24, 4, 256), (16, 8, 256), (16, 1, 512), (16, 4, 128)
    kind = rng.choice(["decode_split", "batch", "batch", "batch_window", "layer", "decode_f32", "tree", "tree", "flash",
                       "prefill", "prefill", "prefill_window", "prefill_chunk", "flash_v2", "flash_v2"])
    kv = rng.choice(["f16", "bf16"])
    if kind == "decode_split":
        heads = rng.choice([q35, slide, small])
        a, k = short(kv, "fp32", size(1, 8), 1, heads, 8191)
    elif kind == "batch":
        heads = rng.choice([q35, q35, slide, glob, small])
        a, k = short(kv, kv, size(1, 16), 1, heads, 8191, chunk=rng.choice([0, 512]))
    elif kind == "batch_window":
        kind = "batch"
        a, k = short(kv, kv, size(1, 16), 1, slide, 16383, chunk=rng.choice([96, 128, 256]), window=rng.choice([512, 1024]))
    elif kind == "layer":
        a, k = short("bf16", "bf16", size(1, 16), 1, slide, 4095, chunk=rng.choice([96, 128, 256]), window=1024)
    elif kind == "decode_f32":
        a, k = short("fp32", "fp32", size(1, 16), 1, rng.choice([q35, slide, small]), 4095)
    elif kind == "tree":
        heads = rng.choice([q35, q35, slide, small])
        a, k = short(kv, kv, size(1, 16), rng.randint(4, 16), heads, 12000, chunk=rng.choice([0, 512, 640]))
    elif kind == "flash":
        n = size(64, 16383)
        a, k = (kv, "fp32", 1, rng.randint(1, 32)) + rng.choice([q35, slide, glob]), dict(lo=n, hi=n)
    elif kind == "prefill":
        heads = rng.choice([q35, slide, slide, glob, small])
        a, k = (kv, kv, 1, size(64, 2048 if heads != glob else 1400)) + heads, dict(lo=0, hi=0)
    elif kind == "prefill_window":
        kind = "prefill"
        a, k = (kv, kv, 1, size(1024, 4096)) + slide, dict(lo=0, hi=0, window=rng.choice([512, 1024]))
    elif kind == "prefill_chunk":
        kind = "prefill"
        n = size(512, 4096)
        a, k = (kv, kv, 1, size(64, 512)) + rng.choice([q35, slide]), dict(lo=n, hi=n, split=rng.choice([-1, 0]))
    else:
        a, k = (kv, "fp32", 1, size(64, 1600)) + rng.choice([q35, slide]), dict(lo=0, hi=0)
    return _case(kind, *a, **k)


# ---------------------------------------------------------------- inputs
def _lens(c):
    """Context lengths before the query tokens, by case."""
    return np.random.default_rng(c["lens"]).integers(c["lo"], c["hi"], size=c["B"], endpoint=True).astype(np.int64)


def _trees(c):
    """Draft trees as ancestor masks: every node has at most two children, parents precede children."""
    r = np.random.default_rng(c["lens"] + 1)
    anc = np.zeros((c["B"], c["T"]), np.uint32)
    for b in range(c["B"]):
        par, kids = [-1], [0] * c["T"]
        for j in range(1, c["T"]):
            p = int(r.choice([p for p in range(j) if kids[p] < 2]))
            par.append(p)
            kids[p] += 1
        for j in range(c["T"]):
            x = j
            while x >= 0:
                anc[b, j] |= np.uint32(1 << x)
                x = par[x]
    return anc


def _inputs(c, seed):
    """The tensors of a case, the same for prepare() and exact()."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)
    lens = _lens(c)
    B, T, NQ, NKV, HD = c["B"], c["T"], c["NQ"], c["NKV"], c["HD"]
    ML = (int(lens.max()) + T + 63) // 64 * 64             # cache rows of a sequence
    kd, qd = DT[c["kv"]], DT[c["io"]]
    sd = 1.0 if c["kind"] in ("prefill", "flash_v2", "layer") else 0.5

    def randn(*shape, dtype=torch.float32):
        return torch.randn(*shape, device="cuda", generator=g, dtype=dtype)

    x = dict(lens=lens, ML=ML, K=randn(B, ML, NKV, HD, dtype=kd).mul_(sd), V=randn(B, ML, NKV, HD, dtype=kd).mul_(sd),
             anc=_trees(c) if c["kind"] == "tree" else None)
    if c["kind"] == "layer":                               # projections before the norm, weights, RoPE tables
        x.update(xq=randn(B, NQ, HD), xk=randn(B, NKV, HD), xv=randn(B, NKV, HD), wq=1 + 0.1 * randn(HD), wk=1 + 0.1 * randn(HD))
        f = 10000.0 ** (-torch.arange(HD // 2, device="cuda", dtype=torch.float64) / (HD // 2))
        ang = torch.arange(ML, device="cuda", dtype=torch.float64)[:, None] * f
        x.update(cos=torch.cat([ang.cos(), ang.cos()], 1).float(), sin=torch.cat([ang.sin(), ang.sin()], 1).float())
    else:
        x["Q"] = randn(B, T, NQ, HD).to(qd)
    return x


def prepare(case, seed):
    c, s = case, _inputs(case, seed)
    B, T, NQ, HD = c["B"], c["T"], c["NQ"], c["HD"]
    lens = s["lens"]
    s["c"] = c
    s["max_pos"] = int(lens.max()) + T - 1
    s["stride"] = s["ML"] * c["NKV"] * HD
    s["pos"] = torch.from_numpy(lens.astype(np.int32)).cuda()        # position of each sequence's first query token
    s["O"] = torch.empty(B, T, NQ, HD, device="cuda", dtype=DT[c["io"]])
    if s["anc"] is not None:
        s["anc"] = torch.from_numpy(s["anc"].reshape(-1).view(np.int32)).cuda()
    if c["kind"] in ("batch", "layer", "tree", "decode_split"):      # the split scratch, once, as a server does at start
        chunk = c["chunk"] or A.split_chunk()
        A.split_reserve(B * T * max(1, -(-A.split_chunk() // chunk)), NQ, s["ML"], HD)
    if c["kind"] == "decode_f32":
        A.flash_reserve_partials(B * NQ * (s["ML"] // 512 + 1), HD)
    if c["kind"] == "flash":
        A.flash_reserve(T, NQ, int(lens[0]), HD)
    if c["kind"] == "layer":
        s["Q"] = torch.empty(B, T, NQ, HD, device="cuda", dtype=DT[c["io"]])
    return s


def run(state):
    s, c = state, state["c"]
    B, T, NQ, NKV, HD, w = c["B"], c["T"], c["NQ"], c["NKV"], c["HD"], c["window"]
    K, V, O = s["K"], s["V"], s["O"]
    kind = c["kind"]
    if kind == "decode_split":
        A.decode_split(s["Q"], K, V, O, B, NQ, NKV, HD, 0, 1, s["pos"], s["max_pos"], s["stride"], A.split_ns_cap(s["ML"]),
                       window=w)
    elif kind in ("batch", "tree"):
        A.attn_batch(s["Q"], K, V, O, B, T, NQ, NKV, HD, s["pos"], s["stride"], s["max_pos"], chunk=c["chunk"], anc=s["anc"],
                     window=w)
    elif kind == "layer":
        code, row = A.kv_code(K), NKV * HD
        A.norm_rope_store(s["xq"], s["wq"], s["Q"], code, B * NQ, NQ, HD, 1e-6, s["cos"], s["sin"], pos_arr=s["pos"],
                          slot_stride=NQ * HD, row_stride=0)
        A.norm_rope_store(s["xk"], s["wk"], K, code, B * NKV, NKV, HD, 1e-6, s["cos"], s["sin"], pos_arr=s["pos"],
                          slot_stride=s["stride"], row_stride=row)
        A.norm_rope_store(s["xv"], None, V, code, B * NKV, NKV, HD, 1e-6, pos_arr=s["pos"], slot_stride=s["stride"],
                          row_stride=row, rope=False)
        A.attn_batch(s["Q"], K, V, O, B, T, NQ, NKV, HD, s["pos"], s["stride"], s["max_pos"], chunk=c["chunk"], window=w)
        return {"O": O, "K": K, "V": V}
    elif kind == "decode_f32":
        A.attn_decode_batch(s["Q"], K, V, O, B, NQ, NKV, HD, 0, s["stride"], window=w, base_b=s["pos"])
    elif kind == "flash":
        A.flash_attn(s["Q"], K, V, O, T, NQ, NKV, HD, c["lo"], window=w)
    elif kind == "flash_v2":
        A.flash_attn_v2(s["Q"], K, V, O, T, NQ, NKV, HD, c["lo"], window=w)
    else:
        A.attn_prefill(s["Q"], K, V, O, B, T, NQ, NKV, HD, base=c["lo"], kv_split=c["split"], window=w)
    return {"O": O}


# ---------------------------------------------------------------- what a pass cannot do without
def _keys(c):
    """Attended (query token, key) pairs, and keys read at least once, over the sequences (one KV head)."""
    anc, pairs, keys, w = (_trees(c) if c["kind"] == "tree" else None), 0, 0, c["window"]
    for b, n in enumerate(_lens(c)):
        pos = n + np.arange(c["T"], dtype=np.int64)
        lo = np.maximum(0, pos - w + 1) if w else np.zeros_like(pos)
        if anc is None:
            pairs += int((pos + 1 - lo).sum())
        else:
            pairs += int(n) * c["T"] + sum(bin(int(a)).count("1") for a in anc[b])
        keys += int(pos[-1] + 1 - lo[0])
    return pairs, keys


def work(case):
    c = case
    pairs, keys = _keys(c)
    rows = c["B"] * c["T"]
    nbytes = keys * c["NKV"] * c["HD"] * 2 * SIZE[c["kv"]] + 2 * rows * c["NQ"] * c["HD"] * SIZE[c["io"]]
    if c["kind"] == "layer":               # fp32 projections in, tables and weights in (the new K and V rows count as keys)
        nbytes += rows * (c["NQ"] + 2 * c["NKV"]) * c["HD"] * 4 + rows * c["HD"] * 4 + 2 * c["HD"] * 4
    return {"bytes": nbytes, "flops": 4 * c["HD"] * c["NQ"] * pairs}


def tolerance(case):
    # About four times the error against exact(): 2.4e-3 with bf16 (Q, or the output, rounded once to 8 bits), 2.9e-4
    # with f16 caches (Q, probabilities and output to 11 bits), 3.2e-7 with fp32 ones (sums only); fp32 sums over
    # thousands of keys in another order move by more than the error of one order, hence ten times there.
    if case["kv"] == "fp32":
        return {"rel": 3e-6}
    return {"rel": 9e-3 if case["kv"] == "bf16" else 1.2e-3}


# ---------------------------------------------------------------- 64-bit results
def _attend(q, k, v, pos, window, anc):
    """q [T, NQ, HD], k / v [n, NKV, HD], all float64; token t at pos[t], tree masks relative to pos[0]."""
    T, NQ, HD = q.shape
    NKV = k.shape[1]
    G = NQ // NKV
    o = torch.empty_like(q)
    for t0 in range(0, T, 512):
        t1 = min(T, t0 + 512)
        p = torch.arange(int(pos[t0]), int(pos[t1 - 1]) + 1, device=q.device)
        j0 = max(0, int(pos[t0]) - window + 1) if window else 0
        j = torch.arange(j0, int(pos[t1 - 1]) + 1, device=q.device)
        ok = j[None, :] <= p[:, None]
        if window:
            ok &= j[None, :] > p[:, None] - window
        if anc is not None:
            d = j - int(pos[0])
            bits = torch.from_numpy(anc[t0:t1].astype(np.int64)).to(q.device)
            ok &= (d < 0)[None, :] | ((bits[:, None] >> d.clamp(0, 31)[None, :]) & 1).bool()
        for h in range(NKV):
            qh = q[t0:t1, h * G:(h + 1) * G].reshape(-1, HD).contiguous()
            s = torch.mm(qh, k[j0:j0 + len(j), h].t().contiguous()) / math.sqrt(HD)
            s.masked_fill_(~ok.repeat_interleave(G, 0), -math.inf)
            o[t0:t1, h * G:(h + 1) * G] = torch.mm(torch.softmax(s, -1), v[j0:j0 + len(j), h].contiguous()).reshape(-1, G, HD)
    return o


def _norm(x, w):
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6)
    return y if w is None else y * w


def _rope(y, cos, sin):
    h = y.shape[-1] // 2
    a, b, c, s = y[..., :h], y[..., h:], cos[:, None, :h], sin[:, None, :h]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def exact(case, seed):
    c, x = case, _inputs(case, seed)
    B, T, NQ, HD = c["B"], c["T"], c["NQ"], c["HD"]
    K, V = x["K"], x["V"]
    if c["kind"] == "layer":
        K, V = K.double(), V.double()
        at = torch.from_numpy(x["lens"]).cuda()
        cos, sin = x["cos"].double()[at], x["sin"].double()[at]
        Q = _rope(_norm(x["xq"].double(), x["wq"].double()), cos, sin)[:, None]
        for b in range(B):
            K[b, at[b]] = _rope(_norm(x["xk"].double(), x["wk"].double()), cos, sin)[b]
            V[b, at[b]] = _norm(x["xv"].double(), None)[b]
    else:
        Q = x["Q"].double()
    O = torch.empty(B, T, NQ, HD, device="cuda", dtype=torch.float64)
    for b in range(B):
        n = int(x["lens"][b])
        O[b] = _attend(Q[b], K[b, :n + T].double(), V[b, :n + T].double(), np.arange(n, n + T), c["window"],
                       None if x["anc"] is None else x["anc"][b])
    return {"O": O, "K": K, "V": V} if c["kind"] == "layer" else {"O": O}
