"""Timing cases: what a program that embeds text and searches the embeddings has
this library do, through the package's public entry points.

Kinds of case (the key "kind"):
  embed      token IDs -> L2-normalized embeddings, the whole 24-layer Q8_0
             model.  "api" is "host" (Model.forward_packed: host token IDs and
             host result, the serving call) or "device" (Model.forward_device:
             both in HBM, the bulk call); "attn" the model's attention mode.
  ffn        the Q8_0 feed-forward block over the kernel seam, for a program
             that adopts the kernels piecewise: RMSNorm, per-sequence int8
             quantization, gate/up + GELUQuick, quantization, down projection.
  attention  the attention layer over the kernel seam (MQA, 3 query heads,
             1 kv head, head_dim 256, bidirectional, ragged sequences).
  search     top-k of a batch of queries against a brute-force index that the
             program keeps.
  index      a brute-force index built from embeddings already in HBM, then
             searched once (what a refresh of a collection does).

Weights are random Q8_0 tensors of the model's shapes and byte format, loaded
once per process, as a serving process does.  exact() restates each path in
64-bit torch arithmetic; int8 quantization, the polynomial exponential and the
fp16 block scales are part of what the path computes and stay in it.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(_ROOT, "go-semantica_amd") not in sys.path:
    sys.path.insert(0, os.path.join(_ROOT, "go-semantica_amd"))

from semantica_gpu import Context, Model, _lib, kernels, search, synth  # noqa: E402

CFG = synth.EMBEDDINGGEMMA_300M
D, FF, HEADS, HD = CFG["embed_dim"], CFG["interm_dim"], CFG["num_heads"], 256
LAYER_WEIGHTS = D * (D + 2 * HD) + D * D + 2 * D * FF + D * FF  # Q8_0 values per layer
Q8_BYTES = 34 / 32  # bytes per Q8_0 value
MODES = {"float32": search.QUANTIZE_FLOAT32, "int8": search.QUANTIZE_INT8, "int16": search.QUANTIZE_INT16}
MODE_BYTES = {"float32": 4, "int8": 1, "int16": 2}


def listed():
    return [
        # One short query on the serving path: launches and latency.
        _embed("embed-1x32", "host", 1, "fixed", 32, 32, 768),
        # A handful of queries of a few words to two sentences each.
        _embed("embed-13-queries", "host", 13, "uniform", 5, 60, 256),
        # One document of an odd length.
        _embed("embed-1x509", "host", 1, "fixed", 509, 509, 512),
        # A mixed batch, lengths log-uniform, Matryoshka-truncated.
        _embed("embed-256-ragged", "device", 256, "log", 8, 512, 256),
        # The throughput batch: documents cut to 512 tokens.
        _embed("embed-64x512", "device", 64, "fixed", 512, 512, 768),
        # Long documents up to the model's context: attention-heavy.
        _embed("embed-8-long", "device", 8, "uniform", 1024, 2048, 768),
        # Embeddings that must equal the reference's bit for bit.
        _embed("embed-20-exact", "device", 20, "uniform", 32, 400, 768, "exact"),
        # Single layers over the kernel seam.
        {"name": "ffn-2048", "kind": "ffn", "rows": 2048, "n": 9},
        {"name": "attention-6-seqs", "kind": "attention", "n": 6, "lo": 300, "hi": 1100},
        # Retrieval: a batch of queries against a million vectors, and one
        # query against a smaller full-precision collection.
        {"name": "search-64q-1M-int8", "kind": "search", "mode": "int8", "count": 1000000, "dim": 768, "q": 64, "k": 10},
        {"name": "search-1q-150k-f32", "kind": "search", "mode": "float32", "count": 150001, "dim": 512, "q": 1, "k": 20},
        # A collection's refresh: index its new embeddings, look a few up.
        {"name": "index-100k-int16", "kind": "index", "mode": "int16", "count": 100000, "dim": 256, "q": 16, "k": 10},
    ]


def _embed(name, api, n, dist, lo, hi, dim, attn="fast"):
    return {"name": name, "kind": "embed", "api": api, "n": n, "dist": dist, "lo": lo, "hi": hi, "dim": dim,
            "attn": attn}


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    pick = rng.random()
    if pick < 0.5:
        attn = "exact" if rng.random() < 0.15 else "fast"
        dim = rng.choice((768, 512, 256, 128))
        shape = rng.random()
        if shape < 0.35:  # queries
            n, lo = _log_int(rng, 1, 48), rng.randint(3, 24)
            c = _embed("", "host", n, "uniform", lo, rng.randint(lo, 64), dim, attn)
        elif shape < 0.75:  # documents
            lo = _log_int(rng, 65, 1024)
            hi = rng.randint(lo, min(2048, 3 * lo))
            most = 5000 if attn == "exact" else 30000 if hi <= 600 else 12000
            n = _log_int(rng, 1, max(1, most // hi))
            c = _embed("", rng.choice(("host", "device")), n, "uniform", lo, hi, dim, attn)
        else:  # mixed
            hi = _log_int(rng, 64, 700)
            n = _log_int(rng, 2, 24 if attn == "exact" else 12000 // hi)
            c = _embed("", "device", n, "log", rng.randint(3, 16), hi, dim, attn)
        del c["name"]
        return c
    if pick < 0.6:
        rows = _log_int(rng, 17, 12000)
        return {"kind": "ffn", "rows": rows, "n": rng.randint(1, min(rows, 40))}
    if pick < 0.7:
        lo = _log_int(rng, 20, 900)
        hi = rng.randint(lo, min(2048, 3 * lo))
        return {"kind": "attention", "n": _log_int(rng, 1, max(1, 9000 // hi)), "lo": lo, "hi": hi}
    mode = rng.choice(("int8", "int8", "int16", "float32"))
    dim = rng.choice((768, 512, 256, 128, rng.randint(65, 767)))
    k = _log_int(rng, 1, 100)
    if pick < 0.92:
        q = _log_int(rng, 1, 100)
        most = min(1000000, 64 * 10**6 * 768 // (q * dim), 10**9 // (dim * MODE_BYTES[mode]))
        return {"kind": "search", "mode": mode, "count": _log_int(rng, 2000, most), "dim": dim, "q": q, "k": k}
    return {"kind": "index", "mode": mode, "count": _log_int(rng, 2000, 200000), "dim": dim,
            "q": _log_int(rng, 1, 32), "k": k}


# ---- what a program keeps ---------------------------------------------------


@functools.lru_cache(maxsize=None)
def _weights():
    return synth.make_model()


@functools.lru_cache(maxsize=None)
def _ctx():
    return Context(0)


@functools.lru_cache(maxsize=None)
def _model(attn):
    m = Model(_ctx(), _weights())
    m.set_attention_mode(_lib.SG_ATTN_EXACT if attn == "exact" else _lib.SG_ATTN_FAST)
    return m


@functools.lru_cache(maxsize=None)
def _ffn_weights():
    ly = _weights().layers[7]
    return {k: kernels.Q8Weight(_ctx(), ly[k], *s) for k, s in
            (("ffn_gate", (FF, D)), ("ffn_up", (FF, D)), ("ffn_down", (D, FF)))}


def _lengths(case, seed):
    if case["dist"] == "fixed":
        return np.full(case["n"], case["lo"], np.int32)
    if case["dist"] == "log":
        return synth.lengths_log_uniform(case["n"], case["lo"], case["hi"], 1)
    return synth.lengths_uniform(case["n"], case["lo"], case["hi"], 4)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))


def _vectors(case, g):
    """Embedding-like vectors: a direction common to all, topics, and noise."""
    n, dim = case["count"], case["dim"]
    common = torch.randn(dim, generator=g, device="cuda")
    topics = torch.randn(500, dim, generator=g, device="cuda")
    which = torch.randint(0, 500, (n,), generator=g, device="cuda")
    v = torch.randn(n, dim, generator=g, device="cuda")
    for i in range(0, n, 1 << 16):
        v[i:i + (1 << 16)] += 0.7 * topics[which[i:i + (1 << 16)]] + 0.5 * common
    near = torch.randint(0, n, (case["q"],), generator=g, device="cuda")
    q = v[near] + 0.8 * torch.randn(case["q"], dim, generator=g, device="cuda")
    return v, q.cpu().numpy()


def _ids(n):
    return (np.arange(n, dtype=np.int64) * 7 + 3).astype(np.int32)


def _activations(rows, cols, g):
    """Hidden-state-like rows: a few columns much larger than the rest."""
    x = torch.randn(rows, cols, generator=g, device="cuda")
    x[:, ::97] *= 8.0
    return x


def _ffn_lengths(case):
    n, rows = case["n"], case["rows"]
    cuts = [rows * (i * i + i) // (n * n + n) for i in range(n + 1)]
    cuts = [max(c, i) for i, c in enumerate(cuts)]
    return np.asarray([min(c, rows - (n - i)) for i, c in enumerate(cuts)], np.int32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "embed":
        off = synth.offsets_from_lengths(_lengths(case, seed))
        toks = synth.token_ids(int(off[-1]), CFG["vocab_size"], seed)
        st = {"case": case, "model": _model(case["attn"]), "off": off, "toks": toks}
        if case["api"] == "device":
            st["d_toks"] = torch.from_numpy(toks).cuda()
            st["out"] = torch.empty(case["n"], case["dim"], device="cuda")
        return st
    g = _gen(seed)
    if kind == "ffn":
        off = _ffn_lengths(case)
        rows = case["rows"]
        ly = _weights().layers[7]
        return {"case": case, "off": off, "w": _ffn_weights(), "x": _activations(rows, D, g),
                "norm": torch.from_numpy(ly["ffn_norm"]).cuda(),
                "lens": torch.from_numpy(np.diff(off).astype(np.int64)).cuda()}
    if kind == "attention":
        off = synth.offsets_from_lengths(synth.lengths_uniform(case["n"], case["lo"], case["hi"], 4))
        t = int(off[-1])
        # QK-normed rows (norm weights near 1) and value rows of GEMM outputs.
        q = torch.nn.functional.normalize(torch.randn(t, HEADS, HD, generator=g, device="cuda"), dim=-1)
        k = torch.nn.functional.normalize(torch.randn(t, HD, generator=g, device="cuda"), dim=-1)
        return {"case": case, "off": off, "q": (16 * q).reshape(t, HEADS * HD).contiguous(), "k": 16 * k,
                "v": torch.randn(t, HD, generator=g, device="cuda") * 3.0,
                "out": torch.empty(t, HEADS * HD, device="cuda")}
    v, q = _vectors(case, g)
    st = {"case": case, "q": q, "ids": _ids(case["count"])}
    if kind == "search":
        torch.cuda.synchronize()
        st["index"] = search.Index.from_device(_ctx(), st["ids"], v.data_ptr(), case["dim"], case["count"],
                                               MODES[case["mode"]])
    else:
        st["v"] = v
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "embed":
        if case["api"] == "host":
            return st["model"].forward_packed(st["toks"], st["off"], case["dim"])
        st["model"].forward_device(st["d_toks"].data_ptr(), st["off"], case["dim"], st["out"].data_ptr())
        return st["out"]
    if kind == "ffn":
        ctx, off, w, x, rows = _ctx(), st["off"], st["w"], st["x"], case["rows"]
        xn = torch.empty_like(x)
        kernels.rmsnorm(ctx, xn, x, st["norm"], CFG["norm_eps"])
        q = torch.empty(rows, D, dtype=torch.int8, device="cuda")
        sc = torch.empty(case["n"], device="cuda")
        kernels.quantize_symmetric_int8(ctx, xn, off, q, sc)
        h = torch.empty(rows, FF, device="cuda")
        kernels.ffn_gate_up(ctx, h, w["ffn_gate"], w["ffn_up"], q,
                            torch.repeat_interleave(sc, st["lens"], output_size=rows))
        q2 = torch.empty(rows, FF, dtype=torch.int8, device="cuda")
        sc2 = torch.empty(case["n"], device="cuda")
        kernels.quantize_symmetric_int8(ctx, h, off, q2, sc2)
        y = torch.empty(rows, D, device="cuda")
        kernels.matmul_q8_0(ctx, y, w["ffn_down"], q2, torch.repeat_interleave(sc2, st["lens"], output_size=rows))
        return {"scale": sc, "h": h, "scale2": sc2, "y": y}
    if kind == "attention":
        kernels.attention(_ctx(), st["out"], st["q"], st["k"], st["v"], HEADS, 1, HD, st["off"])
        return st["out"]
    if kind == "search":
        ids, dist, found = st["index"].search_batch(st["q"], case["k"])
        return {"ids": ids, "dist": dist, "found": found}
    index = search.Index.from_device(_ctx(), st["ids"], st["v"].data_ptr(), case["dim"], case["count"],
                                     MODES[case["mode"]],
                                     stream=torch.cuda.current_stream().cuda_stream)
    ids, dist, found = index.search_batch(st["q"], case["k"])
    index.close()
    return {"ids": ids, "dist": dist, "found": found}


def work(case):
    kind = case["kind"]
    if kind == "embed":
        lens = _lengths(case, 0).astype(np.float64)
        t, L = lens.sum(), CFG["num_layers"]
        return {"bytes": L * LAYER_WEIGHTS * Q8_BYTES + t * (4 + D * Q8_BYTES) + 4.0 * case["n"] * case["dim"],
                "flops": L * (2.0 * t * LAYER_WEIGHTS + 4.0 * HEADS * HD * float((lens * lens).sum()))}
    if kind == "ffn":
        t = case["rows"]
        return {"bytes": 3 * D * FF * Q8_BYTES + 8.0 * t * D + 4.0 * t * FF, "flops": 2.0 * t * 3 * D * FF}
    if kind == "attention":
        lens = synth.lengths_uniform(case["n"], case["lo"], case["hi"], 4).astype(np.float64)
        return {"bytes": 4.0 * lens.sum() * (2 * HEADS + 2) * HD, "flops": 4.0 * HEADS * HD * float((lens * lens).sum())}
    n, dim, q, k = case["count"], case["dim"], case["q"], min(case["k"], case["count"])
    b = n * dim * MODE_BYTES[case["mode"]] + 4.0 * q * dim + 12.0 * q * k
    if kind == "index":
        b += 4.0 * n * dim
    return {"bytes": b, "flops": 2.0 * n * dim * q}


def tolerance(case):
    kind = case["kind"]
    if kind == "embed":
        # 24 layers with four int8 quantizations each: one unit in the last
        # place anywhere flips codes, and the flips compound (0.004 to 0.017
        # from exact()).
        return {"rel": 0.03, "max": 0.5}
    if kind == "ffn":
        return {"rel": 2e-3, "max": 5e-2}  # flipped codes: 2e-4 (h), 5e-4 (y) from exact()
    if kind == "attention":
        return {"rel": 1.2e-5, "max": 1e-3}  # 2.7e-6 from exact()
    return "exact"  # ids and distances are the reference's, bit for bit


# ---- the same in 64 bits ----------------------------------------------------


def _q8(raw, gguf_subnormals=False):
    """Raw Q8_0 blocks [rows, blocks, 34] -> (int8 values, fp64 block scales) on the GPU."""
    t = torch.from_numpy(np.ascontiguousarray(raw)).cuda()
    h = t[..., 0].to(torch.int64) | (t[..., 1].to(torch.int64) << 8)
    d = h.to(torch.int16).view(torch.float16).to(torch.float64)
    if gguf_subnormals:  # the token table's converter halves subnormal scales
        d = torch.where((h & 0x7C00) == 0, d / 2, d)
    return t[..., 2:].contiguous().view(torch.int8), d


def _dense(raw):
    q, d = _q8(raw)
    return (q.to(torch.float64) * d.unsqueeze(-1)).reshape(q.shape[0], -1)


def _seq_of(off):
    return torch.repeat_interleave(torch.arange(len(off) - 1, device="cuda"),
                                   torch.from_numpy(np.diff(off).astype(np.int64)).cuda())


def _quantized(x, seq, n):
    """Symmetric int8 per sequence: (codes as fp64, scale per sequence)."""
    m = torch.zeros(n, dtype=torch.float64, device="cuda").scatter_reduce(0, seq, x.abs().amax(1), "amax")
    s = torch.where(m == 0, torch.ones_like(m), m / 127)
    p = x / s[seq].unsqueeze(1)
    return torch.sign(p) * torch.floor(p.abs() + 0.5), s


def _matmul(x, w, seq, n):
    codes, s = _quantized(x, seq, n)
    return (codes @ w.T) * s[seq].unsqueeze(1)


def _rms(x, w, eps):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y * w


def _fast_exp(x):
    """2^(x log2 e) as exponent and fourth-order polynomial; 0 below -10 (x <= 0)."""
    y = x * 1.442695041
    i = torch.trunc(y)
    f = y - i
    p = 1 + f * (0.693147180559945 + f * (0.240226506959101 + f * (0.055504108664821 + f * 0.009676036358193)))
    return torch.where(x < -10, torch.zeros_like(x), p * torch.exp2(i))


def _gelu_quick(x):
    e = _fast_exp(-(1.702 * x).abs())
    return x * torch.where(x >= 0, torch.ones_like(e), e) / (1 + e)


def _attention(q, k, v, off):
    """q [t, heads, hd], k and v [t, hd]: softmax over each sequence with _fast_exp."""
    out = torch.empty_like(q)
    for a, b in zip(off[:-1], off[1:]):
        a, b = int(a), int(b)
        for h in range(HEADS):
            s = (q[a:b, h] @ k[a:b].T) / math.sqrt(HD)
            e = _fast_exp(s - s.amax(1, keepdim=True))
            out[a:b, h] = (e @ v[a:b]) / e.sum(1, keepdim=True)
    return out


def _rope(x, c, s):
    a, b = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat((a * c - b * s, a * s + b * c), -1)


def _exact_embed(case, seed):
    w = _weights()
    off = synth.offsets_from_lengths(_lengths(case, seed))
    toks = synth.token_ids(int(off[-1]), CFG["vocab_size"], seed)
    n, t = case["n"], int(off[-1])
    seq = _seq_of(off)
    pos = torch.arange(t, device="cuda") - torch.from_numpy(off[:-1].astype(np.int64)).cuda()[seq]
    # The rotation angles are float32 values: position times a float32 frequency.
    freq = (1.0 / torch.pow(torch.tensor(CFG["rope_base"], dtype=torch.float64),
                            torch.arange(0, HD, 2, dtype=torch.float64) / HD)).to(torch.float32).cuda()
    th = (pos.to(torch.float32).unsqueeze(1) * freq).to(torch.float64)
    c, s = torch.cos(th), torch.sin(th)
    f64 = lambda a: torch.from_numpy(a).cuda().to(torch.float64)  # noqa: E731
    eps = CFG["norm_eps"]
    q, d = _q8(w.token_embd[toks], True)
    h = (q.to(torch.float64) * d.unsqueeze(-1)).reshape(t, D) * math.sqrt(D)
    for ly in w.layers:
        x = _rms(h, f64(ly["attn_norm"]), eps)
        qkv = _matmul(x, torch.cat([_dense(ly[k]) for k in ("attn_q", "attn_k", "attn_v")]), seq, n)
        qq = _rms(qkv[:, :D].reshape(t, HEADS, HD), f64(ly["attn_q_norm"]), eps)
        kk = _rms(qkv[:, D:D + HD], f64(ly["attn_k_norm"]), eps)
        qq = _rope(qq, c.unsqueeze(1), s.unsqueeze(1))
        o = _attention(qq, _rope(kk, c, s), qkv[:, D + HD:], off).reshape(t, D)
        h = h + _rms(_matmul(o, _dense(ly["attn_output"]), seq, n), f64(ly["post_attention_norm"]), eps)
        x = _rms(h, f64(ly["ffn_norm"]), eps)
        codes, sc = _quantized(x, seq, n)
        sc = sc[seq].unsqueeze(1)
        g = _gelu_quick((codes @ _dense(ly["ffn_gate"]).T) * sc) * ((codes @ _dense(ly["ffn_up"]).T) * sc)
        h = h + _rms(_matmul(g, _dense(ly["ffn_down"]), seq, n), f64(ly["post_ffw_norm"]), eps)
    x = _rms(h, f64(w.output_norm), eps)
    p = torch.zeros(n, D, dtype=torch.float64, device="cuda").index_add_(0, seq, x)
    p = p / torch.bincount(seq, minlength=n).to(torch.float64).unsqueeze(1)
    p = p[:, :case["dim"]]
    p = p / p.norm(dim=1, keepdim=True)
    return p if case["api"] == "device" else p.cpu().numpy()


def _exact_ffn(case, seed):
    ly = _weights().layers[7]
    off = _ffn_lengths(case)
    seq, n = _seq_of(off), case["n"]
    x = _activations(case["rows"], D, _gen(seed)).to(torch.float64)
    codes, sc = _quantized(_rms(x, torch.from_numpy(ly["ffn_norm"]).cuda().to(torch.float64), CFG["norm_eps"]), seq, n)
    r = sc[seq].unsqueeze(1)
    h = _gelu_quick((codes @ _dense(ly["ffn_gate"]).T) * r) * ((codes @ _dense(ly["ffn_up"]).T) * r)
    codes2, sc2 = _quantized(h, seq, n)
    return {"scale": sc, "h": h, "scale2": sc2, "y": (codes2 @ _dense(ly["ffn_down"]).T) * sc2[seq].unsqueeze(1)}


def _exact_search(case, seed):
    v, q = _vectors(case, _gen(seed))
    q = torch.from_numpy(q).cuda().to(torch.float64)
    q = q / q.norm(dim=1, keepdim=True)
    dots = torch.empty(case["q"], case["count"], dtype=torch.float64, device="cuda")
    steps = {"float32": None, "int8": 127.0, "int16": 32767.0}[case["mode"]]
    for i in range(0, case["count"], 1 << 16):
        x = v[i:i + (1 << 16)].to(torch.float64)
        x = x / x.norm(dim=1, keepdim=True)
        if steps:
            p = x.clamp(-1, 1) * steps
            x = torch.sign(p) * torch.floor(p.abs() + 0.5) / steps
        dots[:, i:i + (1 << 16)] = q @ x.T
    k = min(case["k"], case["count"])
    return {"ids": None, "dist": dots.topk(k, dim=1).values.cpu().numpy(), "found": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "embed":
        return _exact_embed(case, seed)
    if kind == "ffn":
        return _exact_ffn(case, seed)
    if kind == "attention":
        st = prepare(case, seed)
        f = lambda x: x.to(torch.float64)  # noqa: E731
        return _attention(f(st["q"]).reshape(-1, HEADS, HD), f(st["k"]), f(st["v"]), st["off"]).reshape(-1, HEADS * HD)
    return _exact_search(case, seed)
