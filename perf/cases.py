"""The work that programs have this library do, as cases that can be timed
and compared: single tokens through the decoder, chunks of a known text,
whole teacher-forced windows, codec calls on bytes, and CDF tables, each
through the public Python API, on models of several shapes and weight types.

Every result is bit-exact by the library's contract (the reference fixes the
order and rounding of each operation), so every tolerance is "exact".
"""
from __future__ import annotations

import math

import numpy as np
import torch

from detllm_amd import codec, coder, synth
from detllm_amd.gguf import GGML_F32, GGML_Q4_0, GGML_Q4_K, GGML_Q6_K, GGML_Q8_0, GgufWriter
from detllm_amd.model import F32Llama

ESCAPES = 256

# The four workload shapes of detllm_amd.synth, and "wide": a generic decoder
# with 128-wide heads, the head size of most larger models.
SHAPES = {
    name: dict(arch=w.arch, layers=w.layers, d=w.d, heads=w.heads, kv_heads=w.kv_heads, ff=w.ff, vocab=w.vocab,
               rope_base=w.rope_base, eps=w.eps, tied=w.tied, bias=w.qkv_bias)
    for name, w in synth.WORKLOADS.items()
}
SHAPES["wide"] = dict(arch="llama", layers=12, d=1024, heads=8, kv_heads=2, ff=2816, vocab=32000, rope_base=1e4,
                      eps=1e-5, tied=False, bias=False)

# Weight types a shape's matrices allow (Q4_K and Q6_K need widths of whole
# 256-element superblocks).
WEIGHTS = {
    "tiny": ["f32"],
    "smollm2": ["q8_0", "q4_0", "f32"],
    "qwen05": ["q8_0", "q4_0"],
    "tinyllama": ["q4k_mix", "q8_0"],
    "wide": ["q8_0", "q4_0", "q4k_mix", "f32"],
}


def _case(name, call, shape, weights, layers, ctx, pos, n, chunk, vocab=0):
    c = dict(call=call, shape=shape, weights=weights, layers=layers, ctx=ctx, pos=pos, n=n, chunk=chunk,
             vocab=vocab or SHAPES[shape]["vocab"])
    return dict(c, name=name) if name else c


def listed():
    return [
        # One token of the smallest model (the reference's fixture size and
        # type): nothing but launches and latency.
        _case("token-tiny-f32", "token", "tiny", "f32", 2, 8, 5, 1, 3),
        # Interactive decoding with a small Q8_0 model: one token, its logits
        # returned to the caller.
        _case("token-q8-135m", "token", "smollm2", "q8_0", 30, 2048, 301, 1, 64),
        # One symbol of a decompression: forward of the last symbol, CDF,
        # lookup, range decoder; deep in a 2048-token window.
        _case("decode-step-q8-0.5b", "decode", "qwen05", "q8_0", 24, 2048, 1501, 1, 64),
        # One token of the largest configured model, Q4_K / Q6_K weights.
        _case("token-q4k-1.1b", "token", "tinyllama", "q4k_mix", 22, 2048, 700, 1, 64),
        # One token of a model with 128-wide heads and Q4_0 weights, far into
        # a long window.
        _case("token-q4_0-head128", "token", "wide", "q4_0", 12, 4096, 2903, 1, 64),
        # The ragged end of a text: 13 positions left over after whole chunks.
        _case("chunk-13-q8", "chunk", "qwen05", "q8_0", 8, 2048, 1024, 13, 64),
        # A chunk of an unquantised model, off any multiple of the tiles.
        _case("chunk-100-f32", "chunk", "smollm2", "f32", 6, 2048, 57, 100, 128),
        # A prompt in one call, logits of every position returned.
        _case("prompt-512-q4k", "chunk", "tinyllama", "q4k_mix", 22, 2048, 0, 512, 512),
        # A whole window's teacher-forced encode in chunks of 64: the
        # benchmark's workload.
        _case("window-2048-q4k", "window", "tinyllama", "q4k_mix", 22, 2048, 0, 2048, 64),
        # The codec's encoder on a token stream, with the codec's chunk.
        _case("encode-1000-q8", "encode", "qwen05", "q8_0", 24, 2048, 0, 1000, 512),
        # A short file compressed and decompressed again, over several windows.
        _case("file-200-q8", "file", "smollm2", "q8_0", 8, 128, 0, 200, 512),
        # The full CDF table of logits a program holds on the host.
        _case("cdf-table-152k", "cdf", "qwen05", "q8_0", 0, 1, 0, 1, 1),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    call = rng.choice(["token", "token", "token", "decode", "chunk", "chunk", "chunk", "window", "window", "encode",
                       "file", "cdf"])
    shape = rng.choice(["smollm2", "qwen05", "tinyllama", "wide"] + (["tiny"] if call in ("token", "chunk") else []))
    weights = rng.choice(WEIGHTS[shape])
    full = SHAPES[shape]["vocab"]
    vocab = full if rng.random() < 0.5 else _log_int(rng, min(full, 300), full)
    if call == "cdf":
        return _case("", call, "qwen05", "q8_0", 0, 1, 0, 1, 1, _log_int(rng, 256, 151936))
    layers = _log_int(rng, 1, min(8, SHAPES[shape]["layers"]))
    ctx = {"tiny": 256, "wide": 4096}.get(shape, 2048)
    if call in ("token", "decode"):
        n, chunk = 1, 64
    elif call == "chunk":
        n = _log_int(rng, 2, min(ctx // 2, 512))
        chunk = max(n, 64)
    elif call == "file":
        n, chunk, ctx = _log_int(rng, 20, 200), 512, rng.randint(40, 300)
    else:
        n = _log_int(rng, 65, 2048)
        chunk = _log_int(rng, 16, 512)
    pos = _log_int(rng, 1, ctx - n - 1) if call in ("token", "decode", "chunk") else 0
    return _case("", call, shape, weights, layers, ctx, pos, n, chunk, vocab)


# ---- models ---------------------------------------------------------------------

_KINDS = {"f32": GGML_F32, "q8_0": GGML_Q8_0, "q4_0": GGML_Q4_0, "q4_k": GGML_Q4_K, "q6_k": GGML_Q6_K}


def _raw(rng, n):
    return rng.integers(0, 2**64, (n + 7) // 8, dtype=np.uint64).view(np.uint8)[:n]


def _scales(rng, n, sigma):
    # positive f16 scales within a factor of two either way
    return (sigma * (0.5 + 1.5 * rng.random(n, dtype=np.float32))).astype(np.float16).view(np.uint8).reshape(n, 2)


def _matrix(rng, kind, rows, cols, std):
    """Blocks of a rows x cols matrix whose values have about this deviation."""
    if kind == "f32":
        return rng.standard_normal(rows * cols, dtype=np.float32) * np.float32(std)
    if kind == "q8_0":
        b = _raw(rng, rows * cols // 32 * 34).reshape(-1, 34)
        q = b[:, 2:].view(np.int8)
        np.maximum(q, -127, out=q)
        b[:, :2] = _scales(rng, len(b), std / 94)
    elif kind == "q4_0":
        b = _raw(rng, rows * cols // 32 * 18).reshape(-1, 18)
        b[:, :2] = _scales(rng, len(b), std / 6)
    elif kind == "q4_k":  # (d sc) q - dmin m, 6-bit sc and m, q in 0..15
        b = _raw(rng, rows * cols // 256 * 144).reshape(-1, 144)
        s = _scales(rng, len(b), std / 220)
        b[:, 0:2] = s
        b[:, 2:4] = (7.5 * s.view(np.float16).astype(np.float32)).astype(np.float16).view(np.uint8)
    else:  # q6_k: d scale (q - 32)
        b = _raw(rng, rows * cols // 256 * 210).reshape(-1, 210)
        b[:, 208:210] = _scales(rng, len(b), std / 1700)
    return b


def _tensors(case, seed):
    """(name, rows or 0, cols, kind, data) of every tensor, from the seed."""
    s = dict(SHAPES[case["shape"]], vocab=case["vocab"], layers=case["layers"])
    rng = np.random.Generator(np.random.SFC64([seed & 0xFFFFFFFF, 0xDE7]))
    d, ff, hd = s["d"], s["ff"], s["d"] // s["heads"]
    mix = case["weights"] == "q4k_mix"

    def kind(role, layer=1):
        if not mix:
            return case["weights"]
        return "q6_k" if role in ("v", "output") or (role == "down" and layer % 2 == 0) else "q4_k"

    def mat(name, rows, cols, k, gain=1.0):
        return name, rows, cols, k, _matrix(rng, k, rows, cols, gain / math.sqrt(cols))

    def vec(name, n, mean, sigma):
        return name, 0, n, "f32", (rng.standard_normal(n, dtype=np.float32) * sigma + mean).astype(np.float32)

    # A tied embedding is also the output matrix: logits of a few units.
    yield mat("token_embd.weight", s["vocab"], d, kind("embd"), 2.5)
    for l in range(s["layers"]):
        p = f"blk.{l}."
        yield vec(p + "attn_norm.weight", d, 1.0, 0.02)
        yield mat(p + "attn_q.weight", d, d, kind("q"))
        yield mat(p + "attn_k.weight", s["kv_heads"] * hd, d, kind("k"))
        yield mat(p + "attn_v.weight", s["kv_heads"] * hd, d, kind("v"))
        if s["bias"]:
            for nm, n in (("q", d), ("k", s["kv_heads"] * hd), ("v", s["kv_heads"] * hd)):
                yield vec(p + f"attn_{nm}.bias", n, 0.0, 0.02)
        yield mat(p + "attn_output.weight", d, d, kind("o"))
        yield vec(p + "ffn_norm.weight", d, 1.0, 0.02)
        yield mat(p + "ffn_gate.weight", ff, d, kind("gate"))
        yield mat(p + "ffn_up.weight", ff, d, kind("up"))
        yield mat(p + "ffn_down.weight", d, ff, kind("down", l))
    yield vec("output_norm.weight", d, 1.0, 0.02)
    if not s["tied"]:
        yield mat("output.weight", s["vocab"], d, kind("output"), 2.5)


def _gguf(case, seed):
    s = SHAPES[case["shape"]]
    g = GgufWriter()
    g.add_str("general.architecture", s["arch"])
    p = s["arch"] + "."
    for k, v in (("block_count", case["layers"]), ("context_length", case["ctx"]), ("embedding_length", s["d"]),
                 ("feed_forward_length", s["ff"]), ("attention.head_count", s["heads"]),
                 ("attention.head_count_kv", s["kv_heads"]), ("vocab_size", case["vocab"])):
        g.add_u32(p + k, v)
    g.add_f32(p + "rope.freq_base", s["rope_base"])
    g.add_f32(p + "attention.layer_norm_rms_epsilon", s["eps"])
    if case["call"] == "file":  # the codec's byte-fallback vocabulary
        tokens, types = synth.vocabulary(case["vocab"])
        g.add_str_array("tokenizer.ggml.tokens", tokens)
        g.add_i32_array("tokenizer.ggml.token_type", types)
    for name, rows, cols, kind, data in _tensors(case, seed):
        g.add_tensor(name, (cols, rows) if rows else (cols,), _KINDS[kind], data)
    return g.to_bytes()


def _inputs(case, seed):
    """The token ids of positions 0 .. pos + n and what follows them."""
    rng = np.random.Generator(np.random.SFC64([seed & 0xFFFFFFFF, 0x70CE]))
    ranks = np.arange(1, case["vocab"] + 1, dtype=np.float64) ** -1.1  # token frequencies follow Zipf's law
    cdf = np.cumsum(ranks / ranks.sum())
    perm = rng.permutation(case["vocab"])
    ids = np.minimum(np.searchsorted(cdf, rng.random(case["pos"] + case["n"] + 1)), case["vocab"] - 1)
    return perm[ids].astype(np.uint32)


def _host_logits(case, seed):
    rng = np.random.Generator(np.random.SFC64([seed & 0xFFFFFFFF, 0xCDF]))
    return rng.standard_normal(case["vocab"], dtype=np.float32) * np.float32(2.5)


def _text(case, seed):
    return synth.markov_bytes(seed & 0xFFFFFFFF, case["n"])


# ---- the passes -----------------------------------------------------------------

def prepare(case, seed):
    call = case["call"]
    if call == "cdf":
        return {"call": call, "logits": _host_logits(case, seed)}
    data = _gguf(case, seed)
    if call == "file":
        return {"call": call, "model": codec.LoadedModel.load(data), "text": _text(case, seed), "ctx": case["ctx"],
                "chunk": case["chunk"]}
    model = F32Llama.from_gguf(data)
    ids = _inputs(case, seed)
    session = model.forward_workspace(case["ctx"], case["chunk"])
    pos, n = case["pos"], case["n"]
    for p in range(0, pos, case["chunk"]):  # the text before the call
        session.forward_chunk(ids[p:min(pos, p + case["chunk"])], p)
    st = {"call": call, "model": model, "session": session, "pos": pos, "tokens": ids[pos:pos + n],
          "next": ids[pos + 1:pos + n + 1], "rows": np.arange(n, dtype=np.uint32)}
    if call == "decode":  # a payload whose next symbol is the text's
        session.forward_one(int(ids[pos]), pos, want_logits=False)
        cum, freq, total = session.symbol_ranges(st["next"], 0, ESCAPES)
        enc = coder.RangeEncoder()
        enc.encode(int(cum[0]), int(freq[0]), int(total[0]))
        st["payload"] = enc.finish()
    return st


def _padded(data, symbols):
    """Coded bytes in an array whose length does not depend on the text (a
    symbol takes at most four bytes, the header and the flush 64)."""
    out = np.zeros(4 * symbols + 128, np.uint8)
    out[:len(data)] = np.frombuffer(data, np.uint8)
    return out


def run(state):
    call = state["call"]
    if call == "cdf":
        t = coder.logits_to_cdf_with_byte_escapes(state["logits"])
        return {"freq": t.freq, "cum": t.cum, "total": t.total}
    if call == "file":
        file = codec.compress(state["model"], state["text"], state["ctx"], state["chunk"])
        back = codec.decompress(state["model"], file, state["chunk"])
        return {"file": _padded(file, len(state["text"])), "file_bytes": len(file),
                "text": np.frombuffer(back, np.uint8)}
    s = state["session"]
    if call == "token":
        return {"logits": s.forward_one(int(state["tokens"][0]), state["pos"])}
    if call == "decode":
        dec = coder.RangeDecoder(state["payload"])
        symbol = s.forward_decode(int(state["tokens"][0]), state["pos"], dec, ESCAPES)
        return {"symbol": symbol, "logits": s.logits()}
    if call == "chunk":
        return {"logits": s.forward_chunk(state["tokens"], state["pos"], want_logits=True)}
    if call == "window":
        cum, freq, total = s.forward_ranges(state["tokens"], state["pos"], state["rows"], state["next"], ESCAPES)
        return {"cum": cum, "freq": freq, "total": total}
    payload = codec.encode_symbols_with_model(s, state["tokens"], s.n_ctx // 4)
    return {"payload": _padded(payload, len(state["tokens"])), "payload_bytes": len(payload)}


def work(case):
    V = case["vocab"]
    if case["call"] == "cdf":
        return {"bytes": 4 * V + 12 * (V + ESCAPES), "flops": 30 * V}
    s = SHAPES[case["shape"]]
    d, ff, hd, L = s["d"], s["ff"], s["d"] // s["heads"], case["layers"]
    kv = s["kv_heads"] * hd
    per = {"f32": 4.0, "q8_0": 34 / 32, "q4_0": 18 / 32, "q4_k": 144 / 256, "q6_k": 210 / 256}
    mix = case["weights"] == "q4k_mix"
    k = (lambda big: "q6_k" if big else "q4_k") if mix else (lambda big: case["weights"])
    weight_bytes = V * d * per[k(True)]
    for l in range(L):
        weight_bytes += (2 * d * d + kv * d + 2 * ff * d) * per[k(False)] + kv * d * per[k(True)]
        weight_bytes += d * ff * per[k(l % 2 == 0)]
    macs = V * d + L * (2 * d * d + 2 * kv * d + 3 * ff * d)
    n, pos = case["n"], case["pos"]
    if case["call"] == "file":  # each decoded byte is a forward of its own
        keys = n * min(n, case["ctx"]) / 2
        return {"bytes": (n + 2) * weight_bytes + keys * L * 2 * kv * 4,
                "flops": 2 * (3 * n * macs + 3 * keys * L * 2 * d)}
    keys = n * pos + n * (n + 1) / 2
    out = n * V * 4 if case["call"] in ("token", "chunk", "decode") else n * 20
    return {"bytes": weight_bytes + (pos + 2 * n) * L * 2 * kv * 4 + out, "flops": 2 * (n * macs + keys * L * 2 * d)}


def tolerance(case):
    # The order and rounding of every f32 operation are fixed: logits, CDF
    # entries and coded bytes are the same bits on every implementation.
    return "exact"


# ---- the same results in 64 bits, in plain torch ----------------------------------

def _values(kind, rows, cols, data, dev):
    if kind == "f32":
        v = torch.from_numpy(data).to(dev).double()
        return v.reshape(rows, cols) if rows else v
    b = torch.from_numpy(np.ascontiguousarray(data)).to(dev)

    def half(x):
        return x.contiguous().view(torch.float16).double()

    if kind == "q8_0":
        v = half(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()
    elif kind == "q4_0":
        v = half(b[:, :2]) * (torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8)
    elif kind == "q4_k":
        h, q = b[:, 4:16].int(), b[:, 16:].reshape(-1, 4, 32)
        sc = torch.cat([h[:, :4] & 63, (h[:, 8:] & 15) | ((h[:, :4] >> 6) << 4)], 1).double()
        mn = torch.cat([h[:, 4:8] & 63, (h[:, 8:] >> 4) | ((h[:, 4:8] >> 6) << 4)], 1).double()
        q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        v = (half(b[:, :2]) * sc)[:, :, None] * q - (half(b[:, 2:4]) * mn)[:, :, None]
    else:
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
        low = torch.stack([ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4], 2)
        high = torch.cat([(qh >> (2 * i)) & 3 for i in range(4)], 2)
        q = (low | (high << 4)).reshape(-1, 16, 16).double() - 32
        v = half(b[:, 208:])[:, :, None] * b[:, 192:208].contiguous().view(torch.int8).double()[:, :, None] * q
    return v.reshape(rows, cols)


def _quantised(x, kind):
    """The activations a weight type is multiplied with."""
    if kind == "f32":
        return x
    block = 256 if kind == "q6_k" else 32
    b = x.reshape(-1, block)
    scale = (b.abs().amax(1, keepdim=True) / 127).clamp_min(1e-300)
    y = b / scale
    if kind != "q6_k":  # halves away from zero
        return (torch.sign(y) * torch.floor(y.abs() + 0.5) * scale).reshape(x.shape)
    return (torch.round(y) * scale).reshape(x.shape)


def _exact_logits(case, seed, dev):
    s = SHAPES[case["shape"]]
    w = {name: (kind, _values(kind, rows, cols, data, dev)) for name, rows, cols, kind, data in _tensors(case, seed)}
    ids = torch.from_numpy(_inputs(case, seed)[:case["pos"] + case["n"]].astype(np.int64)).to(dev)
    T, H, KV, hd = len(ids), s["heads"], s["kv_heads"], s["d"] // s["heads"]

    def mul(name, x):
        kind, m = w[name]
        return _quantised(x, kind) @ m.T

    def norm(name, x):
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + s["eps"]) * w[name][1]

    angle = torch.arange(T, device=dev).double()[:, None] * \
        s["rope_base"] ** (-torch.arange(0, hd, 2, device=dev).double() / hd)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def rope(x):
        if s["arch"] == "qwen2":  # halves
            a, b = x[..., :hd // 2], x[..., hd // 2:]
            return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)

    later = torch.ones(T, T, dtype=torch.bool, device=dev).triu(1)
    x = w["token_embd.weight"][1][ids]
    for l in range(case["layers"]):
        p = f"blk.{l}."
        h = norm(p + "attn_norm.weight", x)
        q, k, v = (mul(p + f"attn_{c}.weight", h) for c in "qkv")
        if s["bias"]:
            q, k, v = (t + w[p + f"attn_{c}.bias"][1] for t, c in ((q, "q"), (k, "k"), (v, "v")))
        q, k, v = rope(q.reshape(T, H, hd)), rope(k.reshape(T, KV, hd)), v.reshape(T, KV, hd)
        heads = []
        for i in range(H):
            g = i * KV // H
            sc = (q[:, i] @ k[:, g].T.contiguous() / math.sqrt(hd)).masked_fill(later, -math.inf)
            heads.append(torch.softmax(sc, 1) @ v[:, g])
        x = x + mul(p + "attn_output.weight", torch.cat(heads, 1))
        h = norm(p + "ffn_norm.weight", x)
        g, u = mul(p + "ffn_gate.weight", h), mul(p + "ffn_up.weight", h)
        x = x + mul(p + "ffn_down.weight", g * torch.sigmoid(g) * u)
    last = norm("output_norm.weight", x[case["pos"]:])
    return mul("token_embd.weight" if s["tied"] else "output.weight", last)


def exact(case, seed):
    call = case["call"]
    if call == "cdf":
        e = np.exp(np.maximum(_host_logits(case, seed).astype(np.float64) - _host_logits(case, seed).max(), -88.0))
        freq = np.concatenate([np.floor(e / e.sum() * 2.0**24) + 1, np.ones(ESCAPES)])
        cum = np.cumsum(freq)
        return {"freq": freq, "cum": cum - freq, "total": float(cum[-1])}
    if call not in ("token", "chunk", "decode"):
        return None  # whole numbers and bytes of a range coder: no 64-bit value
    with torch.no_grad():
        y = _exact_logits(case, seed, "cuda" if torch.cuda.is_available() else "cpu").cpu().numpy()
    if call == "token":
        return {"logits": y[0]}
    return {"symbol": None, "logits": y} if call == "decode" else {"logits": y}
