"""The work this backend does for its users, as cases that can be timed and checked.

Two kinds of callers exist. relay's engine calls `HipBackend.forward` with a batch of decode
sequences and prefill chunks, and moves KV blocks between workers with `read_kv_layer` /
`write_kv_layer`; other programs call the kernels of the C ABI (`rh_*`) on device buffers of
their own. The listed cases take both, at the shapes of the three models that the benchmark
runs (SmolLM2-135M, TinyLlama-1.1B, Llama-3-8B) from one-token steps to long-context batches.

Whole steps run 1-4 layers of the larger models (every layer does the same work) and keep the
32,000-token vocabulary for all but SmolLM2, so that the layers and not the logits' copy to
the host stand for the step; SmolLM2 runs whole.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from relay_amd import HipBackend, HipOptions, ModelConfig, _lib
from relay_amd.backend import ForwardBatch, SeqChunk
from relay_amd.model import HostWeights, LayerWeights

DEV = "cuda"
BS = 16  # KV block size of every configuration in this repository

# (hidden, intermediate, layers, heads, kv_heads, head_dim, vocab, rope theta, tied, Llama-3 rope scaling)
MODELS = {
    "smollm2": (576, 1536, 30, 9, 3, 64, 49152, 10000.0, True, False),
    "tinyllama": (2048, 5632, 22, 32, 4, 64, 32000, 10000.0, False, False),
    "llama3": (4096, 14336, 32, 32, 8, 128, 32000, 500000.0, False, True),
}
EPS = 1e-5


def listed():
    return [
        # TinyLlama decoding 32 sequences at 2048 positions: one layer's decode attention.
        {"name": "decode_attn_tinyllama_32x2048", "kind": "decode_attention", "model": "tinyllama", "seqs": 32,
         "ctx": 2048, "ragged": False},
        # Llama-3-8B serving 48 sequences of different lengths up to 8192: one layer's decode attention.
        {"name": "decode_attn_llama3_48x8192", "kind": "decode_attention", "model": "llama3", "seqs": 48, "ctx": 8192,
         "ragged": True},
        # A whole 2048-token TinyLlama prompt in one chunk: one layer's prefill attention.
        {"name": "prefill_attn_tinyllama_2048", "kind": "prefill_attention", "model": "tinyllama", "chunks": 1,
         "rows": 2048, "start": 0},
        # The last 512-token chunk of an 8192-token Llama-3-8B prompt: chunked prefill over a long prefix.
        {"name": "prefill_attn_llama3_512_at_7680", "kind": "prefill_attention", "model": "llama3", "chunks": 1,
         "rows": 512, "start": 7680},
        # One-token int8 projection of Llama-3-8B (gate or up): interactive decoding.
        {"name": "gemv_int8_4096x14336_t1", "kind": "gemv_int8", "tokens": 1, "k": 4096, "n": 14336},
        # The int8 down projection of Llama-3-8B for a mixed batch of 560 tokens.
        {"name": "gemm_int8_14336x4096_t560", "kind": "gemm_int8", "tokens": 560, "k": 14336, "n": 4096},
        # One user chatting with SmolLM2-135M: a whole one-token step, launch- and latency-bound.
        {"name": "step_smollm2_decode_1x640", "kind": "step", "model": "smollm2", "layers": 30, "int8": False,
         "decode": 1, "ctx": 640, "chunk": 0, "start": 0},
        # TinyLlama decode batch: 32 sequences around 2048 positions.
        {"name": "step_tinyllama_decode_32x2048", "kind": "step", "model": "tinyllama", "layers": 4, "int8": False,
         "decode": 32, "ctx": 2048, "chunk": 0, "start": 0},
        # The second 512-token chunk of a TinyLlama prompt (relay's chunked prefill).
        {"name": "step_tinyllama_chunk512_at_512", "kind": "step", "model": "tinyllama", "layers": 4, "int8": False,
         "decode": 0, "ctx": 0, "chunk": 512, "start": 512},
        # Llama-3-8B continuous batching under a 512-token budget: 48 decoding sequences and a prompt chunk.
        {"name": "step_llama3_mixed_48_464", "kind": "step", "model": "llama3", "layers": 2, "int8": False, "decode": 48,
         "ctx": 2048, "chunk": 464, "start": 0},
        # TinyLlama with int8 weights decoding for a few users.
        {"name": "step_tinyllama_int8_decode_8x1024", "kind": "step", "model": "tinyllama", "layers": 4, "int8": True,
         "decode": 8, "ctx": 1024, "chunk": 0, "start": 0},
        # Prefill/decode disaggregation: one layer of an 8192-position Llama-3-8B sequence out of the
        # cache to host memory and into other blocks.
        {"name": "kv_io_llama3_8192", "kind": "kv_io", "model": "llama3", "positions": 8192},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode_attention", "prefill_attention", "gemv_int8", "gemm_int8", "step", "step", "kv_io"])
    model = rng.choice(sorted(MODELS))
    if kind == "decode_attention":
        return {"kind": kind, "model": model, "seqs": _log_int(rng, 1, 48), "ctx": _log_int(rng, 16, 8192),
                "ragged": rng.random() < 0.5}
    if kind == "prefill_attention":
        return {"kind": kind, "model": model, "chunks": rng.choice([1, 1, 2, 3]), "rows": _log_int(rng, 2, 1024),
                "start": rng.choice([0, _log_int(rng, 1, 4096)])}
    if kind == "gemv_int8":
        return {"kind": kind, "tokens": _log_int(rng, 1, 16), "k": 16 * _log_int(rng, 36, 896), "n": _log_int(rng, 500, 14336)}
    if kind == "gemm_int8":
        return {"kind": kind, "tokens": _log_int(rng, 17, 1024), "k": 64 * _log_int(rng, 9, 160), "n": 4 * _log_int(rng, 144, 2048)}
    if kind == "kv_io":
        return {"kind": kind, "model": model, "positions": _log_int(rng, 16, 8192)}
    shape = rng.choice(["decode", "prefill", "mixed"])
    layers = 1 if model == "llama3" else 2
    return {"kind": "step", "model": model, "layers": layers, "int8": rng.random() < 0.4,
            "decode": 0 if shape == "prefill" else _log_int(rng, 1, 48), "ctx": _log_int(rng, 16, 2048),
            "chunk": 0 if shape == "decode" else _log_int(rng, 2, 464 if model == "llama3" else 1024),
            "start": rng.choice([0, _log_int(rng, 1, 1024)])}


# ---- inputs from a seed -------------------------------------------------------------------

def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1000003 + salt)


def _randn(g, *shape, std=1.0):
    """fp32 values that fp16 holds exactly."""
    return (torch.randn(*shape, generator=g, device=DEV) * std).half().float()


def _perm(seed, n):
    return np.random.default_rng(seed).permutation(n).astype(np.int32)


def _contexts(seed, seqs, ctx, ragged):
    """Positions held by each decoding sequence (the token being decoded included)."""
    if not ragged:
        return [ctx] * seqs
    r = np.random.default_rng(seed + 17)
    return [int(v) for v in r.integers(max(1, ctx // 8), ctx + 1, size=seqs)]


def _pool(seed, layer, nblocks, kvh, d):
    """One layer's paged K and V, [block][kv head][slot][dim] fp16."""
    g = _gen(seed, 7 + layer)
    k = torch.randn(nblocks, kvh, BS, d, generator=g, device=DEV, dtype=torch.float16)
    v = torch.randn(nblocks, kvh, BS, d, generator=g, device=DEV, dtype=torch.float16)
    return k, v


def _decode_layout(case, seed):
    ctxs = _contexts(seed, case["seqs"], case["ctx"], case["ragged"])
    lens = [-(-c // BS) for c in ctxs]
    offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    return ctxs, offs, _perm(seed, int(offs[-1]))


def _prefill_layout(case, seed):
    end = case["start"] + case["rows"]
    per = -(-end // BS)
    chunks = [(s * case["rows"], case["rows"], case["start"], s * per) for s in range(case["chunks"])]
    return chunks, per, _perm(seed, per * case["chunks"])


def _step_layout(case, seed):
    """Chunks of the step as (start position, tokens), their block tables and the pool size."""
    vocab = MODELS[case["model"]][6]
    r = np.random.default_rng(seed + 3)
    chunks = []
    if case["decode"]:
        for c in _contexts(seed, case["decode"], case["ctx"], case["decode"] > 1):
            chunks.append((c - 1, r.integers(0, vocab, size=1).tolist()))
    if case["chunk"]:
        chunks.append((case["start"], r.integers(0, vocab, size=case["chunk"]).tolist()))
    lens = [-(-(s + len(t)) // BS) for s, t in chunks]
    nb = sum(lens)
    ids, tables, at = _perm(seed, nb).tolist(), [], 0
    for n in lens:
        tables.append(ids[at:at + n])
        at += n
    return chunks, tables, nb


def _config(case):
    H, I, _, heads, kvh, d, vocab, theta, tied, llama3 = MODELS[case["model"]]
    extra = dict(rope_llama3=True, rope_factor=8.0, rope_low_freq_factor=1.0, rope_high_freq_factor=4.0,
                 rope_original_max_position=8192.0) if llama3 else {}
    return ModelConfig(hidden=H, intermediate=I, layers=case["layers"], heads=heads, kv_heads=kvh, head_dim=d, vocab=vocab,
                       rms_eps=EPS, rope_theta=theta, tie_embeddings=tied, **extra)


def _weights(case, seed):
    """(name, tensor) of every weight, fp32 on the GPU: matrices ~ N(0, 0.02), norms around 1."""
    H, I, _, heads, kvh, d, vocab, _, tied, _ = MODELS[case["model"]]
    g = _gen(seed, 1)
    yield "embed", _randn(g, vocab, H, std=0.02)
    yield "final_norm", 1.0 + _randn(g, H, std=0.1)
    if not tied:
        yield "lm_head", _randn(g, vocab, H, std=0.02)
    for l in range(case["layers"]):
        p = f"layers.{l}."
        yield p + "attn_norm", 1.0 + _randn(g, H, std=0.1)
        yield p + "wqkv", _randn(g, (heads + 2 * kvh) * d, H, std=0.02)
        yield p + "wo", _randn(g, H, heads * d, std=0.02)
        yield p + "mlp_norm", 1.0 + _randn(g, H, std=0.1)
        yield p + "w_gate_up", _randn(g, 2 * I, H, std=0.02)
        yield p + "w_down", _randn(g, H, I, std=0.02)


def _int8(case, seed):
    """Quantized weights of a single product: int8 [N, K] and fp32 row scales; fp16 x."""
    g = _gen(seed)
    w = (torch.randn(case["n"], case["k"], generator=g, device=DEV) * 30).round().clamp(-127, 127).to(torch.int8)
    scale = torch.rand(case["n"], generator=g, device=DEV) * 4e-4 + 4e-4
    x = torch.randn(case["tokens"], case["k"], generator=g, device=DEV).half()
    return w, scale, x


# ---- the cases ----------------------------------------------------------------------------

def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_decode_attention(case, seed):
    heads, kvh, d = MODELS[case["model"]][3:6]
    L = _lib.lib()
    ctxs, offs, ids = _decode_layout(case, seed)
    n = case["seqs"]
    k, v = _pool(seed, 0, len(ids), kvh, d)
    q = torch.randn(n, heads * d, generator=_gen(seed, 2), device=DEV, dtype=torch.float16)
    meta = torch.from_numpy(np.array([[i, c, o, 0] for i, (c, o) in enumerate(zip(ctxs, offs))], np.int32)).to(DEV)
    group = heads // kvh
    slice_keys = L.rh_decode_slice_keys(n, kvh, group, d, max(ctxs))
    parts = -(-max(ctxs) // slice_keys)
    return {"run": _run_decode_attention, "q": q, "k": k, "v": v, "meta": meta, "tables": torch.from_numpy(ids).to(DEV),
            "shape": (n, heads, kvh, d), "slice": slice_keys, "parts": parts,
            "part_o": torch.empty(n * heads * parts * d, device=DEV), "part_ml": torch.empty(n * heads * parts * 2, device=DEV),
            "counters": torch.zeros(n * kvh * (-(-group // 16)), dtype=torch.int32, device=DEV),
            "out": torch.empty(n, heads * d, device=DEV, dtype=torch.float16)}


def _run_decode_attention(s):
    n, heads, kvh, d = s["shape"]
    _lib.check(_lib.lib().rh_paged_decode_attention(
        s["q"].data_ptr(), heads * d, s["k"].data_ptr(), s["v"].data_ptr(), s["meta"].data_ptr(), s["tables"].data_ptr(), n,
        heads, kvh, d, BS, s["slice"], s["parts"], 1.0 / math.sqrt(d), s["part_o"].data_ptr(), s["part_ml"].data_ptr(),
        s["counters"].data_ptr(), s["out"].data_ptr(), heads * d, torch.cuda.current_stream().cuda_stream), "decode attention")
    return s["out"]


def _prepare_prefill_attention(case, seed):
    heads, kvh, d = MODELS[case["model"]][3:6]
    chunks, _, ids = _prefill_layout(case, seed)
    k, v = _pool(seed, 0, len(ids), kvh, d)
    rows = case["rows"] * case["chunks"]
    q = torch.randn(rows, heads * d, generator=_gen(seed, 2), device=DEV, dtype=torch.float16)
    work = torch.from_numpy(_lib.prefill_work(chunks, heads)).to(DEV)
    return {"run": _run_prefill_attention, "q": q, "k": k, "v": v, "tables": torch.from_numpy(ids).to(DEV), "work": work,
            "shape": (heads, kvh, d), "out": torch.empty_like(q)}


def _run_prefill_attention(s):
    heads, kvh, d = s["shape"]
    _lib.check(_lib.lib().rh_flash_prefill(
        s["q"].data_ptr(), heads * d, s["k"].data_ptr(), s["v"].data_ptr(), s["tables"].data_ptr(), s["work"].data_ptr(),
        s["work"].shape[0], heads, kvh, d, BS, 1.0 / math.sqrt(d), s["out"].data_ptr(), heads * d,
        torch.cuda.current_stream().cuda_stream), "prefill attention")
    return s["out"]


def _prepare_int8(case, seed):
    L = _lib.lib()
    w, scale, x = _int8(case, seed)
    ldw = L.rh_gemv_int8_row_stride(case["k"])
    padded = torch.zeros(case["n"], ldw, dtype=torch.int8, device=DEV)
    padded[:, :case["k"]] = w
    return {"w": padded, "ldw": ldw, "scale": scale, "x": x, "shape": (case["tokens"], case["k"], case["n"]),
            "y": torch.empty(case["tokens"], case["n"], device=DEV)}


def _prepare_gemv_int8(case, seed):
    return {"run": _run_gemv_int8, **_prepare_int8(case, seed)}


def _run_gemv_int8(s):
    t, k, n = s["shape"]
    _lib.check(_lib.lib().rh_gemv_int8(s["w"].data_ptr(), s["ldw"], s["scale"].data_ptr(), 0, s["x"].data_ptr(),
                                       s["y"].data_ptr(), t, k, n, 0.0, torch.cuda.current_stream().cuda_stream), "gemv int8")
    return s["y"]


def _prepare_gemm_int8(case, seed):
    s = {"run": _run_gemm_int8, **_prepare_int8(case, seed)}
    ks = _lib.lib().rh_gemm_w8_plan(case["tokens"], case["k"], case["n"])
    s["ksplit"], s["ws"] = ks, torch.empty(ks * case["tokens"] * case["n"] if ks > 1 else 1, device=DEV)
    return s


def _run_gemm_int8(s):
    t, k, n = s["shape"]
    _lib.check(_lib.lib().rh_gemm_w8_split(s["w"].data_ptr(), s["ldw"], s["scale"].data_ptr(), s["x"].data_ptr(),
                                           s["y"].data_ptr(), t, k, n, 0.0, s["ksplit"], s["ws"].data_ptr(),
                                           torch.cuda.current_stream().cuda_stream), "gemm int8")
    return s["y"]


def _prepare_step(case, seed):
    c = _config(case)
    chunks, tables, nb = _step_layout(case, seed)
    tokens = sum(len(t) for _, t in chunks)
    opts = HipOptions(False, case["int8"])
    if case["int8"]:
        host = {name: t.cpu().numpy() for name, t in _weights(case, seed)}
        layers = [LayerWeights(*(host.get(f"layers.{l}.{f}") for f in
                                 ("attn_norm", "wqkv", "bqkv", "wo", "mlp_norm", "w_gate_up", "w_down"))) for l in range(c.layers)]
        w = HostWeights(c, host["embed"], layers, host["final_norm"], host.get("lm_head"))
        be = HipBackend(w, nb, BS, max_batch_tokens=tokens, max_context=nb * BS, options=opts)
    else:
        be = HipBackend(None, nb, BS, max_batch_tokens=tokens, max_context=nb * BS, options=opts, config=c, synthetic_seed=0)
        for name, t in _weights(case, seed):
            torch.cuda.synchronize()
            be.update_weight(name, t)
    for l in range(c.layers):
        kv = torch.cat([t.flatten().view(torch.uint8) for t in _pool(seed, l, nb, c.kv_heads, c.head_dim)])
        be.write_kv_layer(l, list(range(nb)), kv.cpu().numpy())
    batch = ForwardBatch([SeqChunk(t, s, tab, True) for (s, t), tab in zip(chunks, tables)])
    return {"run": _run_step, "backend": be, "batch": batch}


def _run_step(s):
    return s["backend"].forward(s["batch"])


def _prepare_kv_io(case, seed):
    c = _config({"model": case["model"], "layers": 2})
    n = -(-case["positions"] // BS)
    nb = 2 * n
    be = HipBackend(None, nb, BS, max_batch_tokens=16, max_context=nb * BS, options=HipOptions(False, False), config=c,
                    synthetic_seed=0)
    kv = torch.cat([t.flatten().view(torch.uint8) for t in _pool(seed, 0, n, c.kv_heads, c.head_dim)]).cpu().numpy()
    ids = _perm(seed, nb).tolist()
    out = np.full(kv.size, 255, np.uint8)
    return {"run": _run_kv_io, "backend": be, "data": kv, "blocks": ids[:n], "out": out}


def _run_kv_io(s):
    be = s["backend"]
    be.write_kv_layer(1, s["blocks"], s["data"])
    return be.read_kv_layer(1, s["blocks"], out=s["out"])


# ---- work, tolerance ------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "decode_attention":
        heads, kvh, d = MODELS[case["model"]][3:6]
        # a ragged batch holds 9/16 of its longest context on average
        keys = case["seqs"] * case["ctx"] * (0.5625 if case["ragged"] else 1.0)
        return {"bytes": keys * kvh * d * 4 + 4 * case["seqs"] * heads * d, "flops": 4.0 * keys * heads * d}
    if kind == "prefill_attention":
        heads, kvh, d = MODELS[case["model"]][3:6]
        rows, start, n = case["rows"], case["start"], case["chunks"]
        pairs = n * (rows * start + rows * (rows + 1) / 2)
        return {"bytes": n * (4 * rows * heads * d + (start + rows) * kvh * d * 4), "flops": 4.0 * pairs * heads * d}
    if kind in ("gemv_int8", "gemm_int8"):
        t, k, n = case["tokens"], case["k"], case["n"]
        return {"bytes": n * k + 4 * n + 2 * t * k + 4 * t * n, "flops": 2.0 * t * k * n}
    H, I, _, heads, kvh, d, vocab, _, tied, _ = MODELS[case["model"]]
    if kind == "kv_io":
        b = -(-case["positions"] // BS) * BS * kvh * d * 4
        return {"bytes": 4 * b, "flops": 0}  # each direction reads and writes the blocks once
    dec, chunk, start = case["decode"], case["chunk"], case["start"]
    tokens, rows = dec + chunk, dec + (1 if chunk else 0)
    params = (heads + 2 * kvh) * d * H + H * heads * d + 3 * H * I
    keys = dec * case["ctx"] * (0.5625 if dec > 1 else 1.0)
    pairs = keys + chunk * start + chunk * (chunk + 1) / 2
    by = case["layers"] * (params * (1 if case["int8"] else 2) + (keys + start + tokens) * kvh * d * 4)
    return {"bytes": by + 2 * vocab * H + 2 * tokens * H + 4 * rows * vocab,
            "flops": case["layers"] * (2.0 * tokens * params + 4.0 * pairs * heads * d) + 2.0 * rows * vocab * H}


def tolerance(case):
    kind = case["kind"]
    if kind == "kv_io":
        return "exact"
    if kind in ("gemv_int8", "gemm_int8"):
        return {"rel": 2e-6}  # fp32 sums of exact products, up to 14336 terms (4e-7 off 64 bits)
    if kind in ("decode_attention", "prefill_attention"):
        return {"rel": 1.5e-3}  # fp16 queries, softmax weights and outputs (3e-4 off 64 bits)
    # fp16 activations through the layers (1e-3 off 64 bits over 1-4 layers, 2e-3 over 30)
    return {"rel": 8e-3 if case["layers"] > 4 else 4e-3}


# ---- the same outputs in 64 bits ------------------------------------------------------------

def _gather(pool, table, length):
    """Rows 0 .. length of a sequence, [position, kv head, dim] in float64."""
    t = torch.as_tensor(table, dtype=torch.int64, device=DEV)
    kvh, d = pool.shape[1], pool.shape[3]
    return pool[t].permute(0, 2, 1, 3).reshape(-1, kvh, d)[:length].double()


def _attend(q, k, v, start):
    """q [rows, heads, d] at positions start.., k / v [keys, kv heads, d]: causal attention."""
    rows, heads, d = q.shape
    keys, kvh, _ = k.shape
    out = torch.empty_like(q)
    mask = torch.arange(keys, device=DEV)[None, :] > (start + torch.arange(rows, device=DEV))[:, None]
    for h in range(heads):
        kh = h // (heads // kvh)
        s = (q[:, h] @ k[:, kh].T.contiguous()) / math.sqrt(d)
        out[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), dim=-1) @ v[:, kh].contiguous()
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "kv_io":
        return None
    return globals()["_exact_" + kind](case, seed)


def _exact_decode_attention(case, seed):
    heads, kvh, d = MODELS[case["model"]][3:6]
    ctxs, offs, ids = _decode_layout(case, seed)
    k, v = _pool(seed, 0, len(ids), kvh, d)
    q = torch.randn(case["seqs"], heads * d, generator=_gen(seed, 2), device=DEV, dtype=torch.float16).double()
    out = []
    for i, c in enumerate(ctxs):
        tab = ids[offs[i]:offs[i + 1]]
        kk, vv = _gather(k, tab, c), _gather(v, tab, c)
        qi = q[i].view(kvh, heads // kvh, d)
        s = torch.matmul(qi, kk.permute(1, 2, 0).contiguous()) / math.sqrt(d)
        out.append(torch.matmul(torch.softmax(s, -1), vv.permute(1, 0, 2).contiguous()).reshape(-1))
    return torch.stack(out)


def _exact_prefill_attention(case, seed):
    heads, kvh, d = MODELS[case["model"]][3:6]
    chunks, per, ids = _prefill_layout(case, seed)
    k, v = _pool(seed, 0, len(ids), kvh, d)
    rows, end = case["rows"], case["start"] + case["rows"]
    q = torch.randn(rows * case["chunks"], heads * d, generator=_gen(seed, 2), device=DEV, dtype=torch.float16).double()
    out = [_attend(q[t0:t0 + n].view(n, heads, d), _gather(k, ids[off:off + per], end), _gather(v, ids[off:off + per], end), p0)
           for t0, n, p0, off in chunks]
    return torch.cat(out).reshape(rows * case["chunks"], heads * d)


def _exact_gemv_int8(case, seed):
    w, scale, x = _int8(case, seed)
    return (x.double() @ w.double().T) * scale.double()


_exact_gemm_int8 = _exact_gemv_int8


def _inv_freq(case):
    d, theta, llama3 = MODELS[case["model"]][5], MODELS[case["model"]][7], MODELS[case["model"]][9]
    out = []
    for i in range(0, d, 2):
        f = theta ** (-i / d)
        if llama3:  # wavelengths past the original context are stretched 8x, the middle band blended
            low, high, factor, orig = 1.0, 4.0, 8.0, 8192.0
            wavelen = 2 * math.pi / f
            if wavelen > orig / low:
                f = f / factor
            elif wavelen >= orig / high:
                smooth = (orig / wavelen - low) / (high - low)
                f = (1 - smooth) * f / factor + smooth * f
        out.append(f)
    return torch.tensor(out, dtype=torch.float64, device=DEV).float().double()  # the tables hold fp32


def _exact_step(case, seed):
    H, I, _, heads, kvh, d, vocab, _, tied, _ = MODELS[case["model"]]
    chunks, tables, nb = _step_layout(case, seed)
    it = _weights(case, seed)
    embed = next(it)[1].double()
    final_norm = next(it)[1].double()
    head = embed if tied else next(it)[1].double()

    def norm(x, w):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w

    def matrix(w):
        if not case["int8"]:
            return w.double()
        scale = w.abs().amax(1, keepdim=True) / 127.0
        return (w / scale).round().clamp(-127, 127).double() * scale.double()

    tok = torch.tensor([t for _, ts in chunks for t in ts], dtype=torch.int64, device=DEV)
    pos = torch.tensor([s + i for s, ts in chunks for i in range(len(ts))], dtype=torch.float64, device=DEV)
    x = embed[tok]
    ang = pos[:, None] * _inv_freq(case)[None, :]
    cos, sin = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]

    def rope(a):
        lo, hi = a[..., :d // 2], a[..., d // 2:]
        return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin], -1)

    for l in range(case["layers"]):
        an, wqkv, wo, mn, gu, down = (next(it)[1] for _ in range(6))
        pk, pv = _pool(seed, l, nb, kvh, d)
        qkv = norm(x, an.double()) @ matrix(wqkv).T
        q = rope(qkv[:, :heads * d].view(-1, heads, d))
        k = rope(qkv[:, heads * d:(heads + kvh) * d].view(-1, kvh, d))
        v = qkv[:, (heads + kvh) * d:].view(-1, kvh, d)
        outs, t0 = [], 0
        for (start, ts), tab in zip(chunks, tables):
            n = len(ts)
            kk = torch.cat([_gather(pk, tab, start), k[t0:t0 + n]])
            vv = torch.cat([_gather(pv, tab, start), v[t0:t0 + n]])
            if n == 1:
                s = torch.matmul(q[t0].view(kvh, heads // kvh, d), kk.permute(1, 2, 0).contiguous()) / math.sqrt(d)
                outs.append(torch.matmul(torch.softmax(s, -1), vv.permute(1, 0, 2).contiguous()).reshape(1, heads, d))
            else:
                outs.append(_attend(q[t0:t0 + n], kk, vv, start))
            t0 += n
        x = x + torch.cat(outs).reshape(-1, heads * d) @ matrix(wo).T
        g = norm(x, mn.double()) @ matrix(gu).T
        x = x + (torch.nn.functional.silu(g[:, :I]) * g[:, I:]) @ matrix(down).T
    ends = np.cumsum([len(ts) for _, ts in chunks]) - 1
    return norm(x[torch.as_tensor(ends, device=DEV)], final_norm) @ head.T
