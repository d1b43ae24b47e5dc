"""The work a user of this package has it do, as measurable cases.

A retrieval system calls the package in two phases.  Indexing embeds passages and documents in
batches, packs the chunk embeddings, assigns token embeddings to k-means centres and codes the
residuals.  Searching embeds a short query, scores it against the centres and the coded residuals
and unpacks candidate chunks.  Each case below is one such call at one size, through the public
entry points of `witchcraft_amd`; `draw` gives further sizes of the same ranges.

Inputs come from the seed alone.  The encoder's weights are a program's long-lived state: one
random-init XTR-base model per weight layout, laid out once per process and shared by every state,
as one program's encoder serves all of its inputs.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from witchcraft_amd import _lib, codec, score, synth
from witchcraft_amd.encoder import T5EncoderModel

DEV = "cuda:0"
CFG = synth.XTR_BASE
DIM = CFG["proj_dim"]          # columns of every embedding
MODEL_SEED = 20
NUMERICS = {"default": _lib.T5H_NUMERICS_DEFAULT, "hybrid": _lib.T5H_NUMERICS_HYBRID,
            "hybrid_bf16": _lib.T5H_NUMERICS_HYBRID_BF16}
WINDOW, STRIDE = 2048, 256     # Embedder's window and overlap


# ---- the cases -----------------------------------------------------------------------------

def _encode(seqs, lo, hi, lens, api="device", layout="q4k", numerics="default"):
    return {"op": "encode", "seqs": seqs, "lo": lo, "hi": hi, "lens": lens, "api": api, "layout": layout,
            "numerics": numerics}


def listed():
    return [
        # A search box's query: one sequence of 32 tokens, host buffers in and out.
        {"name": "query", **_encode(1, 32, 32, 0, api="host")},
        # One passage of odd length, embedded on its own as it arrives (an indexer without a queue).
        {"name": "passage", **_encode(1, 181, 181, 0, api="host")},
        # The headline batch: 32 sequences of 32 to 256 tokens, resident in device memory.
        {"name": "batch", **_encode(32, 32, 256, 2)},
        # Bulk indexing: 256 passages of 64 to 512 tokens.
        {"name": "bulk", **_encode(256, 64, 512, 4)},
        # The hybrid-dequant build's numerics (with bf16 dense weights, its x86 default).
        {"name": "hybrid", **_encode(64, 16, 512, 5, layout="hybrid", numerics="hybrid_bf16")},
        # Whole documents through overlapping windows, with the norm filter, host buffers.
        {"name": "documents", "op": "embed", "docs": 12, "lo": 10, "hi": 5000, "lens": 6},
        # A query's tokens against the index's centres, the first step of a search.
        {"name": "centre_scores", "op": "scores", "rows": 32, "cols": 16384},
        # The same query against a million coded residuals.
        {"name": "residual_scores", "op": "q4_scores", "rows": 32, "cols": 1048576},
        # k-means assignment of sampled token embeddings when the index is built.
        {"name": "assign", "op": "assign", "rows": 131072, "cols": 16384},
        # Residual codes of the indexed token embeddings.
        {"name": "residual_codes", "op": "encode_residuals", "rows": 1000003, "cols": 16384},
        # Chunk embeddings into the stored form (indexing) and back (search).
        {"name": "pack", "op": "pack", "chunks": 48, "lo": 64, "hi": 512, "lens": 7},
        {"name": "unpack", "op": "unpack", "chunks": 48, "lo": 64, "hi": 512, "lens": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["query", "passage", "batch", "batch", "bulk", "hybrid", "documents", "scores", "q4_scores",
                       "assign", "encode_residuals", "pack", "unpack"])
    lens = rng.randrange(1 << 20)
    if kind == "query":  # up to 64 tokens in one to three short sequences
        n = rng.randint(1, 3)
        return _encode(n, 4, 64 // n, lens, api="host")
    if kind == "passage":
        n = _log_int(rng, 65, 2048)
        return _encode(1, n, n, lens, api="host")
    if kind == "batch":
        hi = rng.choice([64, 128, 256, 512])
        return _encode(_log_int(rng, 2, 96), hi // 8, hi, lens)
    if kind == "bulk":
        hi = rng.choice([200, 256, 333, 512])
        return _encode(_log_int(rng, 64, 256), hi // 8, hi, lens)
    if kind == "hybrid":
        hi = rng.choice([128, 256, 512])
        return _encode(_log_int(rng, 1, 64), max(2, hi // 32), hi, lens, layout="hybrid",
                       numerics=rng.choice(["hybrid", "hybrid_bf16", "default"]))
    if kind == "documents":
        return {"op": "embed", "docs": _log_int(rng, 1, 16), "lo": 10, "hi": _log_int(rng, 500, 5000), "lens": lens}
    if kind in ("scores", "q4_scores"):
        return {"op": kind, "rows": rng.randint(4, 64), "cols": _log_int(rng, 1000, 1048576)}
    if kind == "assign":
        return {"op": kind, "rows": _log_int(rng, 4096, 131072), "cols": _log_int(rng, 256, 16384)}
    if kind == "encode_residuals":
        return {"op": kind, "rows": _log_int(rng, 1000, 1048576), "cols": _log_int(rng, 64, 16384)}
    hi = rng.choice([100, 256, 512, 1500])
    return {"op": kind, "chunks": _log_int(rng, 1, 48 if hi <= 512 else 20), "lo": hi // 8, "hi": hi, "lens": lens}


# ---- inputs --------------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _image(layout):
    return synth.make_model(CFG, seed=MODEL_SEED, layout=layout)


@functools.lru_cache(maxsize=None)
def _model(layout, numerics):
    m = T5EncoderModel.from_gguf(_image(layout), dict(CFG), hip_device=0)
    m.set_numerics(NUMERICS[numerics])
    return m


def _lens(case, n):
    return np.random.default_rng(case["lens"]).integers(case["lo"], case["hi"] + 1, n)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _unit(x):
    return x / x.norm(dim=1, keepdim=True)


def _chunk(r, rows):
    """Token embeddings of one chunk: unit rows that drift around a common direction."""
    x = r.normal(0, 1, DIM) + np.cumsum(r.normal(0, 0.15, (rows, DIM)), axis=0) + r.normal(0, 0.3, (rows, DIM))
    return (x / np.linalg.norm(x, axis=1, keepdims=True)).astype(np.float32)


def prepare(case, seed):
    op = case["op"]
    s = {"op": op, "case": case}
    if op == "encode":
        s["model"] = _model(case["layout"], case["numerics"])
        cu = np.zeros(case["seqs"] + 1, np.int32)
        cu[1:] = np.cumsum(_lens(case, case["seqs"]))
        s["cu"], T = cu, int(cu[-1])
        s["ids"] = np.random.default_rng(seed).integers(1, CFG["vocab_size"], T).astype(np.uint32)
        if case["api"] == "device":
            s["d_ids"] = torch.from_numpy(s["ids"].view(np.int32)).to(DEV)
            s["out"] = torch.empty((T, DIM), device=DEV)
            s["norm"] = torch.empty(T, device=DEV)
    elif op == "embed":
        s["model"] = _model("q4k", "default")
        r = np.random.default_rng(seed)
        s["docs"] = [r.integers(1, CFG["vocab_size"], n).astype(np.uint32) for n in _lens(case, case["docs"])]
    elif op in ("pack", "unpack"):
        r = np.random.default_rng(seed)
        lens = _lens(case, case["chunks"])
        s["mats"] = [_chunk(r, n) for n in lens]
        if op == "unpack":
            s["bufs"] = codec.embeddings_to_packed_batch(s.pop("mats"))
        else:  # where the packed chunks are gathered, as a store's write buffer: room for the largest result
            s["store"] = np.zeros(int(2 * lens.sum() * DIM + 1024 * len(lens)), np.uint8)
    else:
        g, M, N = _gen(seed), case["rows"], case["cols"]
        if op in ("scores", "q4_scores"):
            s["q"] = _unit(torch.randn((M, DIM), device=DEV, generator=g))
            s["out"] = torch.empty((M, N), device=DEV)
            if op == "scores":
                s["b"] = _unit(torch.randn((N, DIM), device=DEV, generator=g))
            else:  # codes of normal residuals: bell-shaped over the 16 levels
                c = (7.5 + 3.5 * torch.randn((N, DIM), device=DEV, generator=g)).round().clamp(0, 15).to(torch.uint8)
                s["codes"] = (c[:, 0::2] * 16 + c[:, 1::2]).contiguous()
        else:  # token embeddings scattered around their cluster's direction
            c = torch.randn((N, DIM), device=DEV, generator=g)
            at = torch.randint(0, N, (M,), device=DEV, generator=g)
            s["emb"] = _unit(c[at] / math.sqrt(DIM) + 0.06 * torch.randn((M, DIM), device=DEV, generator=g))
            s["centres"] = _unit(c + 0.5 * torch.randn((N, DIM), device=DEV, generator=g))
            if op == "assign":
                s["out"] = torch.empty(M, dtype=torch.int32, device=DEV)
            else:
                s["at"] = at.to(torch.int32)
                s["out"] = torch.empty((M, DIM // 2), dtype=torch.uint8, device=DEV)
                s["bad"] = torch.zeros(1, dtype=torch.int32, device=DEV)
    return s


# ---- one pass ------------------------------------------------------------------------------

def run(s):
    op = s["op"]
    if op == "encode":
        m = s["model"]
        if s["case"]["api"] == "host":
            return m.encode_packed(s["ids"], s["cu"], normalize=True)
        m.encode_device(s["d_ids"].data_ptr(), s["cu"], s["out"].data_ptr(), s["norm"].data_ptr())
        m.synchronize()  # the outputs are ready, and the error flag read, only then
        return s["out"], s["norm"]
    if op == "embed":
        return [list(d) for d in s["model"].embed_batch(s["docs"], WINDOW, STRIDE)]
    if op == "pack":
        packed = codec.embeddings_to_packed_batch(s["mats"])
        joined = np.frombuffer(b"".join(packed), np.uint8)
        s["store"][:joined.size] = joined
        return s["store"], np.array([len(p) for p in packed])
    if op == "unpack":
        return codec.embeddings_from_packed_batch(s["bufs"], DIM)
    M, N = s["case"]["rows"], s["case"]["cols"]
    stream = torch.cuda.current_stream().cuda_stream
    if op == "scores":
        score.matmul_t_device(s["q"].data_ptr(), M, s["b"].data_ptr(), N, DIM, s["out"].data_ptr(), stream=stream)
    elif op == "q4_scores":
        codec.matmul_t_q4_device(s["q"].data_ptr(), M, s["codes"].data_ptr(), N, DIM, s["out"].data_ptr(), stream)
    elif op == "assign":
        score.matmul_argmax_device(s["emb"].data_ptr(), M, s["centres"].data_ptr(), N, DIM, s["out"].data_ptr(),
                                   stream=stream)
    else:
        codec.residual_encode_device(s["emb"].data_ptr(), M, s["centres"].data_ptr(), N, s["at"].data_ptr(), DIM,
                                     s["out"].data_ptr(), s["bad"].data_ptr(), stream)
        return s["out"], s["bad"]
    return s["out"]


def _windows(n):
    """Embedder's windows of a document of n tokens: [start, end) pairs."""
    got, start = [], 0
    while True:
        end = min(start + WINDOW, n)
        got.append((start, end))
        if end == n:
            return got
        start += WINDOW - STRIDE


def work(case):
    op = case["op"]
    if op in ("encode", "embed"):
        D, F, inner, layers = CFG["d_model"], CFG["d_ff"], CFG["num_heads"] * CFG["d_kv"], CFG["num_layers"]
        if op == "encode":
            lens = _lens(case, case["seqs"])
            out_rows = int(lens.sum())
        else:
            docs = _lens(case, case["docs"])
            lens = np.array([e - b for n in docs for b, e in _windows(int(n))])
            out_rows = int(docs.sum())
        T = int(lens.sum())
        dense, wi, proj = layers * (4 * D * inner + D * F), layers * 2 * D * F, DIM * D
        q4 = 144 / 256
        dense_bytes = 4.0 if case.get("layout") == "hybrid" else q4
        return {"bytes": dense * dense_bytes + (wi + proj) * q4 + 4.0 * T * (1 + D) + 4.0 * out_rows * (DIM + 1),
                "flops": 2.0 * T * (dense + wi + proj) + 4.0 * inner * layers * float((lens.astype(np.float64) ** 2).sum())}
    if op in ("pack", "unpack"):
        values = float(_lens(case, case["chunks"]).sum()) * DIM
        return {"bytes": values * (4 + 1.7 / 8), "flops": values * 14}
    M, N = case["rows"], case["cols"]
    if op == "scores":
        return {"bytes": 4.0 * (M * DIM + N * DIM + M * N), "flops": 2.0 * M * N * DIM}
    if op == "q4_scores":
        return {"bytes": 4.0 * M * DIM + N * DIM / 2 + 4.0 * M * N, "flops": 2.0 * M * N * DIM}
    if op == "assign":
        return {"bytes": 4.0 * (M * DIM + N * DIM + M), "flops": 2.0 * M * N * DIM}
    return {"bytes": M * (4.0 * DIM + 4 + DIM / 2) + 4.0 * min(M, N) * DIM, "flops": 5.0 * M * DIM}


def tolerance(case):
    op = case["op"]
    if op in ("encode", "embed"):
        # f16 operands in every product of 12 layers: 8e-4 off the 64-bit result by default.  The
        # hybrid numerics round activations to 8 bits per block, and a value that f16 attention
        # moves over a rounding boundary lands one step (1/128 of its block's largest) away: 1e-2.
        return {"rel": 3e-2, "max": 1.0 - 1e-6} if case.get("numerics", "default") != "default" else {"rel": 3e-3, "max": 0.1}
    if op in ("scores", "q4_scores"):
        return {"rel": 1e-6, "max": 1e-5}   # 128-term f32 sums
    if op == "assign":
        return {"differ": 1e-5}             # two centres equally near within f32 rounding
    return "exact"                          # stored bytes, and rows decoded from them


# ---- the same in 64 bits -------------------------------------------------------------------

def _q4k_values(raw, shape):
    """GGML Q4_K super-blocks -> float64: (d * scale) * q - dmin * min per 32 values."""
    b = np.frombuffer(raw, np.uint8).reshape(-1, 144)
    d, dmin = (b[:, i:i + 2].copy().view(np.float16).astype(np.float64) for i in (0, 2))
    p = b[:, 4:16].astype(np.int64)
    lo, mid, hi = p[:, 0:4], p[:, 4:8], p[:, 8:12]
    sc = np.concatenate([lo & 63, (hi & 15) | (lo >> 6 << 4)], 1)
    mn = np.concatenate([mid & 63, (hi >> 4) | (mid >> 6 << 4)], 1)
    qs = b[:, 16:].reshape(-1, 4, 1, 32)
    q = np.concatenate([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
    return ((d * sc)[:, :, None] * q - (dmin * mn)[:, :, None]).reshape(shape)


@functools.lru_cache(maxsize=1)
def _weights(layout):
    """name -> float64 tensor on the GPU of every tensor of the GGUF image."""
    img = _image(layout)
    u32 = lambda p: int.from_bytes(img[p:p + 4], "little")  # noqa: E731
    u64 = lambda p: int.from_bytes(img[p:p + 8], "little")  # noqa: E731
    count, pos, infos, got = u64(8), 24, [], {}
    for _ in range(count):
        n = u64(pos)
        name, pos = img[pos + 8:pos + 8 + n].decode(), pos + 8 + n
        dims = [u64(pos + 4 + 8 * i) for i in range(u32(pos))]
        pos += 4 + 8 * len(dims)
        infos.append((name, dims[::-1], u32(pos), u64(pos + 4)))
        pos += 12
    base = (pos + 31) // 32 * 32
    for name, shape, kind, off in infos:
        n = math.prod(shape)
        if kind == 12:
            v = _q4k_values(img[base + off:base + off + n // 256 * 144], shape)
        else:
            v = np.frombuffer(img, np.float32, n, base + off).astype(np.float64).reshape(shape)
        got[name] = torch.from_numpy(v).to(DEV)
    return got


def _buckets(n):
    """[n, n] relative-position buckets of (query i, key j)."""
    half, far = CFG["relative_attention_num_buckets"] // 2, CFG["relative_attention_max_distance"]
    exact_to = half // 2
    rel = np.arange(n)[None, :] - np.arange(n)[:, None]
    dist = np.abs(rel)
    ratio = np.maximum(dist, 1).astype(np.float32) / np.float32(exact_to)
    big = np.log(ratio) / np.float32(math.log(far / exact_to)) * np.float32(half - exact_to)
    b = np.where(dist < exact_to, dist, np.minimum(exact_to + np.maximum(big, 0).astype(np.int64), half - 1))
    return b + np.where(rel > 0, half, 0)


def _to_q8k(x):
    """Rows rounded as 256-value blocks of 8-bit codes: scale -128 / (first value of largest size)."""
    b = x.reshape(-1, 256)
    top = b.gather(1, b.abs().argmax(1, keepdim=True))
    k = torch.where(top == 0, torch.zeros_like(top), -128.0 / top)
    q = torch.sign(b) * torch.sign(k) * torch.floor((k * b).abs() + 0.5)
    return torch.where(k == 0, torch.zeros_like(b), q.clamp(max=127.0) / k).reshape(x.shape)


def _gelu(x, pade):
    if not pade:
        return torch.nn.functional.gelu(x, approximate="tanh")
    t = (0.7978845608 * x * (1 + 0.044715 * x * x)).clamp(-4.97, 4.97)
    t2 = t * t
    th = t * (135135 + t2 * (17325 + t2 * (378 + t2))) / (135135 + t2 * (62370 + t2 * (3150 + 28 * t2)))
    return 0.5 * x * (1 + th)


def _encode64(layout, numerics, seqs):
    """Un-normalised [L, 128] projections of each id sequence, in float64."""
    w, hybrid = _weights(layout), numerics != "default"
    H, dk, eps = CFG["num_heads"], CFG["d_kv"], CFG["layer_norm_epsilon"]
    # bf16 by truncation of the f32 weight's bits
    cut = ((lambda t: (t.float().view(torch.int32) & -65536).view(torch.float32).double())
           if numerics == "hybrid_bf16" else (lambda t: t))
    q8 = _to_q8k if hybrid else (lambda t: t)
    norm = lambda x, g: x / torch.sqrt((x * x).mean(1, keepdim=True) + eps) * g  # noqa: E731
    lens = [len(i) for i in seqs]
    ids = torch.from_numpy(np.concatenate(seqs).astype(np.int64)).to(DEV)
    rel = w["encoder.block.0.layer.0.SelfAttention.relative_attention_bias.weight"]
    bias = rel[torch.from_numpy(_buckets(max(lens))).to(DEV)].permute(2, 0, 1).contiguous()
    x = w["encoder.embed_tokens.weight"][ids]
    for i in range(CFG["num_layers"]):
        p = "encoder.block.%d.layer." % i
        dense = lambda k: cut(w[p + k + ".weight"]).T.contiguous()  # noqa: E731
        h = norm(x, w[p + "0.layer_norm.weight"])
        q, k, v = (h @ dense("0.SelfAttention." + c) for c in "qkv")
        at, b = [], 0
        for n in lens:
            qs, ks, vs = (t[b:b + n].reshape(n, H, dk).transpose(0, 1).contiguous() for t in (q, k, v))
            a = torch.softmax(torch.matmul(qs, ks.transpose(1, 2).contiguous()) + bias[:, :n, :n], -1)
            at.append(torch.matmul(a, vs).transpose(0, 1).reshape(n, H * dk))
            b += n
        x = x + torch.cat(at) @ dense("0.SelfAttention.o")
        h = q8(norm(x, w[p + "1.layer_norm.weight"]))
        f = p + "1.DenseReluDense."
        g = _gelu(h @ w[f + "wi_0.weight"].T, hybrid) * (h @ w[f + "wi_1.weight"].T)
        x = x + g @ dense("1.DenseReluDense.wo")
    return (q8(norm(x, w["encoder.final_layer_norm.weight"])) @ w["linear.weight"].T).split(lens)


def _argmax64(a, b):
    return torch.cat([(p.double() @ b.double().T).argmax(1) for p in a.split(8192)]).to(torch.int32)


def exact(case, seed):
    op = case["op"]
    if op in ("pack", "unpack", "encode_residuals"):
        return None  # bytes fixed by the format, and rows decoded from them
    s = prepare(case, seed)
    if op == "encode":
        seqs = [s["ids"][a:b] for a, b in zip(s["cu"], s["cu"][1:])]
        y = torch.cat(_encode64(case["layout"], case["numerics"], seqs))
        n = y.norm(dim=1)
        return (y / n[:, None] if case["api"] == "host" else y), n
    if op == "embed":
        spans = [(d, b, e) for d, ids in enumerate(s["docs"]) for b, e in _windows(len(ids))]
        sums = [torch.zeros((len(d), DIM), dtype=torch.float64, device=DEV) for d in s["docs"]]
        for (d, b, e), y in zip(spans, _encode64("q4k", "default", [s["docs"][d][b:e] for d, b, e in spans])):
            sums[d][b:e] += y
        got = []
        for y in sums:  # tokens whose summed embedding is shorter than 1 are dropped
            n = y.norm(dim=1)
            keep = torch.nonzero(n >= 1.0).flatten()
            got.append([_unit(y[keep]), keep.to(torch.int32)])
        return got
    if op == "scores":
        return s["q"].double() @ s["b"].double().T
    if op == "q4_scores":  # the format's 16 levels are f32 values: mu-law, mu = 255, scale 1/4
        x = (np.arange(16, dtype=np.float32) - np.float32(7.5)) * np.float32(2 / 15)
        p = np.exp(np.abs(x) * np.log(np.float32(256)))
        levels = np.sign(x) * ((p - np.float32(1)) * np.float32(1 / 255)) * np.float32(0.25)
        t = torch.from_numpy(levels.astype(np.float64)).to(DEV)
        c = s["codes"]
        r = torch.stack([t[(c >> 4).long()], t[(c & 15).long()]], 2).reshape(c.shape[0], DIM)
        return s["q"].double() @ r.T
    return _argmax64(s["emb"], s["centres"])
