"""The work that users of this framework have it do, as timed cases.

Each case is one call (or one short sequence of calls) through a public entry
point of the package, on inputs of the sizes and distributions of the
repository's benchmark configurations, tests and defaults:

  forward      LMTransformer.forward_with_embeddings, the full entropy model
               (14 layers, dim 768, FFN 2048, vocab 260) on byte tokens
  block        one transformer layer of the same model (a 1-layer
               extract_embeddings): embedding, QKV + RoPE, attention, O, FFN
  attention    fused_attention on bf16 tensors (head_dim 64, matrix cores)
  attention32  fused_attention on f32 tensors (any head_dim)
  entropy      EntropyPatchPlan: logits -> entropies and two boundary rules
  patches      patch_boundaries and patch_means of given entropies
  row_ops      fused_rms_norm (+ L2 norms) and fused_silu_gate of one FFN input
  pipeline     process_document: the chunked streaming loop over one document
  ingest       StreamingIngest over byte documents: packed rows, boundaries,
               per-patch means, host memory in and out

exact() restates every kind in 64-bit torch or numpy, without the package.
"""
import importlib
import math

import numpy as np
import torch

_pkg = importlib.import_module("blt-burn_amd")


def _mod(name):
    return importlib.import_module("blt-burn_amd." + name)


DIM, HEADS, HIDDEN, VOCAB, LAYERS = 768, 12, 2048, 260, 14
MAX_TOKENS = 16 * 8192  # the model handle's bound: a [16, 8192] batch
WEIGHT_SEED = 4
DEV = "cuda"


def listed():
    return [
        # a short string (a title, a chat line): the smallest model call, where
        # weights, latency and launches count
        dict(name="forward_short", kind="forward", batch=1, seq=48, window=512),
        # one default-sized chunk (BltConfig.max_seq_len = 1024)
        dict(name="forward_doc", kind="forward", batch=1, seq=1024, window=512),
        # the full batch of the benchmark's configuration 4
        dict(name="forward_batch", kind="forward", batch=16, seq=8192, window=512),
        # one layer with the reference's full causal attention, ragged length
        dict(name="block_causal", kind="block", batch=2, seq=3001, window=0),
        # configuration 3: windowed attention with RoPE
        dict(name="attention_window", kind="attention", batch=8, heads=12, seq=4096, window=512,
             theta=10000.0),
        # the reference's f32 attention op
        dict(name="attention_f32", kind="attention32", batch=2, heads=12, seq_q=1000, seq_kv=1000,
             head_dim=64, causal=True),
        # configuration 1: entropies and the global and monotonic boundaries
        dict(name="entropy_patches", kind="entropy", batch=4, seq=8192, vocab=260),
        # boundaries and per-patch means of a batch's entropies
        dict(name="patch_means", kind="patches", batch=16, seq=8192),
        # configuration 2: RMSNorm + L2 norms, then SiLU * gate, in bf16
        dict(name="row_ops", kind="row_ops", rows=32768, dim=768, hidden=2048, dtype="bf16"),
        # one document of three chunks through the streaming pipeline
        dict(name="pipeline_document", kind="pipeline", bytes=9000),
        # one document of the default process_bytes configuration
        dict(name="ingest_document", kind="ingest", documents=1, mix=1, chunk=1024,
             overlap=512),
        # many documents packed into 8192-token rows (configuration 5)
        dict(name="ingest_documents", kind="ingest", documents=64, mix=2, chunk=8192,
             overlap=512),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["forward", "forward", "block", "block", "attention", "attention32",
                       "entropy", "patches", "row_ops", "pipeline", "ingest"])
    if kind in ("forward", "block"):
        n = _log(rng, 4, MAX_TOKENS)
        batch = rng.choice([1, 1, 2, 3, 5, 8, 16])
        seq = max(1, min(8192, n // batch))
        window = rng.choice([512, 512, 0])
        # full causal rows cost more per token: at most what a windowed batch costs
        if window == 0:
            batch = max(1, min(batch, 32768 // seq))
        return dict(kind=kind, batch=batch, seq=seq, window=window)
    if kind == "attention":
        seq = _log(rng, 1, 8192)
        batch = max(1, min(rng.choice([1, 2, 3, 8]), 32768 // seq))
        return dict(kind=kind, batch=batch, heads=rng.choice([1, 4, 12]), seq=seq,
                    window=rng.choice([0, 512, 300]), theta=rng.choice([0.0, 10000.0]))
    if kind == "attention32":
        seq_q, d = _log(rng, 1, 2048), rng.choice([32, 64, 64, 80, 128])
        seq_kv = seq_q if rng.random() < 0.6 else _log(rng, 1, 2048)
        heads = rng.choice([2, 4, 12])
        batch = max(1, min(rng.choice([1, 2, 4]), int(2e10 // (4 * seq_q * seq_kv * d * heads))))
        return dict(kind=kind, batch=batch, heads=heads, seq_q=seq_q, seq_kv=seq_kv, head_dim=d,
                    causal=rng.random() < 0.6)
    if kind == "entropy":
        n, batch = _log(rng, 64, 65536), rng.choice([1, 2, 4, 7])
        return dict(kind=kind, batch=batch, seq=max(1, n // batch),
                    vocab=rng.choice([260, 260, 256, 261]))
    if kind == "patches":
        batch = rng.choice([1, 1, 3, 16])
        return dict(kind=kind, batch=batch, seq=max(1, _log(rng, 64, MAX_TOKENS) // batch))
    if kind == "row_ops":
        return dict(kind=kind, rows=_log(rng, 1, 65536), dim=rng.choice([768, 768, 512, 1000, 2048]),
                    hidden=rng.choice([2048, 768, 1001]), dtype=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "pipeline":
        return dict(kind=kind, bytes=_log(rng, 16, 24000))
    return dict(kind=kind, documents=_log(rng, 1, 24), mix=rng.randrange(10000),
                chunk=rng.choice([1024, 2048, 8192]), overlap=rng.choice([256, 512]))


# ---- inputs -------------------------------------------------------------------

_weights = {}
_models = {}


def _get_weights(layers):
    # N(0, 0.02) weights, norm weights 1 + N(0, 0.02), as the benchmark draws them
    if layers not in _weights:
        M = _mod("model")
        cfg = M.entropy_model_config()
        cfg.n_layers = layers
        _weights[layers] = (cfg, M.random_weights(cfg, WEIGHT_SEED, hidden=HIDDEN))
    return _weights[layers]


def _model(layers, window):
    """The model handle a program loads once and keeps."""
    if (layers, window) not in _models:
        cfg, w = _get_weights(layers)
        _models[layers, window] = _mod("model").LMTransformer(
            cfg, w, device=torch.cuda.current_device(), max_tokens=MAX_TOKENS, window=window)
    return _models[layers, window]


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed & 0x7FFFFFFF)
    return g


def _randn(g, shape, dtype=torch.float32, mean=0.0, std=1.0):
    return (torch.randn(shape, generator=g, device=DEV) * std + mean).to(dtype)


def _tokens(case, seed):
    return _mod("synth").tokens(seed & 0x7FFFFFFF, (case["batch"], case["seq"]))


def _document(case, seed):
    return (_mod("synth").tokens(seed & 0x7FFFFFFF, (case["bytes"],)) - 4).astype(np.uint8)


def _doc_offsets(case):
    """Log-normal document lengths (median 2 KB, at least 256 B; no longer than
    16 KB here so that a case's cost follows its number of documents): the
    case's own, whatever the seed, so that outputs have one shape."""
    z = _mod("synth").normal_f32(0x5EED + case["mix"], (case["documents"],))
    lens = np.clip(np.round(2048 * np.exp(z.astype(np.float64))), 256, 16384).astype(np.int64)
    return np.concatenate([np.zeros(1, np.int64), np.cumsum(lens)])


def _documents(case, seed):
    off = _doc_offsets(case)
    return _mod("synth").tokens(seed & 0x7FFFFFFF, (int(off[-1]),)), off


ENTROPY_RULES = ((1, 1.33), (0, 0.2))  # global threshold, monotonic delta


def _entropy64(x):
    lsm = torch.log_softmax(x.double(), -1)
    return -(lsm.exp() * lsm).sum(-1)


def _logits(case, seed):
    """N(0, 2) logits; rows whose entropy or entropy step lies within 1e-3 of a
    threshold are scaled off it, so every correct result has the same starts."""
    x = _randn(_gen(seed), (case["batch"], case["seq"], case["vocab"]), std=2.0)
    for _ in range(50):
        H = _entropy64(x)
        near = (H - ENTROPY_RULES[0][1]).abs() < 1e-3
        near[:, 1:] |= (H[:, 1:] - H[:, :-1] - ENTROPY_RULES[1][1]).abs() < 1e-3
        if not bool(near.any()):
            break
        x = torch.where(near[..., None], x * 1.03, x)
    return x


def _signals(case, seed):
    """Entropies spread as a trained model's on text, and embedding norms."""
    g, shape = _gen(seed), (case["batch"], case["seq"])
    H = (torch.randn(shape, generator=g, device=DEV) * 0.8 + 3.0).clamp_(0.05, 5.5)
    return H, _randn(g, shape, mean=20.0, std=3.0).abs()


def _attention_inputs(case, seed):
    g, dt = _gen(seed), torch.bfloat16
    shape = (case["batch"], case["heads"], case["seq"], 64)
    return [_randn(g, shape, dt) for _ in range(3)]


def _attention32_inputs(case, seed):
    g = _gen(seed)
    b, h, d = case["batch"], case["heads"], case["head_dim"]
    return [_randn(g, (b, h, n, d)) for n in (case["seq_q"], case["seq_kv"], case["seq_kv"])]


def _row_inputs(case, seed):
    g = _gen(seed)
    dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    x = _randn(g, (1, case["rows"], case["dim"]), dt)
    w = _randn(g, (case["dim"],), dt, mean=1.0, std=0.02)
    a, b = (_randn(g, (1, case["rows"], case["hidden"]), dt) for _ in range(2))
    return x, w, a, b


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("forward", "block"):
        m = _model(LAYERS if kind == "forward" else 1, case["window"])
        return dict(case, model=m, tokens=torch.from_numpy(_tokens(case, seed)).to(DEV))
    if kind == "attention":
        return dict(case, qkv=_attention_inputs(case, seed))
    if kind == "attention32":
        return dict(case, qkv=_attention32_inputs(case, seed))
    if kind == "entropy":
        plan = _mod("patcher").EntropyPatchPlan(case["batch"], case["seq"], case["vocab"],
                                                list(ENTROPY_RULES))
        for out in plan.outs:  # entries past a row's count stay as they are
            for t in out:
                t.zero_()
        return dict(case, plan=plan, logits=_logits(case, seed))
    if kind == "patches":
        H, N = _signals(case, seed)
        i32 = dict(dtype=torch.int32, device=DEV)
        shape = tuple(H.shape)
        return dict(case, H=H, N=N,
                    out=tuple(torch.zeros(shape, **i32) for _ in range(3))
                    + (torch.zeros(shape[:1], **i32),),
                    means=(torch.zeros_like(H), torch.zeros_like(H), None))
    if kind == "row_ops":
        x, w, a, b = _row_inputs(case, seed)
        return dict(case, x=x, w=w, a=a, b=b,
                    l2=torch.empty((1, case["rows"]), dtype=torch.float32, device=DEV))
    if kind == "pipeline":
        return dict(case, model=_model(LAYERS, 512), data=_document(case, seed).tobytes())
    tok, off = _documents(case, seed)
    I = _mod("ingest")
    cfg = I.BltConfig(max_seq_len=case["chunk"], chunk_overlap=case["overlap"])
    return dict(case, ingest=I.ingest_for(_model(LAYERS, 512), cfg), tokens=tok, offsets=off)


PATCH_DELTA = 1.335  # BltConfig.threshold


def run(s):
    kind = s["kind"]
    if kind == "forward":
        o = s["model"].forward_with_embeddings(s["tokens"])
        return [o.logits, o.pre_norm_embeddings, o.embedding_norms, o.entropies,
                o.coherence_scores]
    if kind == "block":
        return s["model"].extract_embeddings(s["tokens"])
    if kind == "attention":
        q, k, v = s["qkv"]
        return _mod("fused_ops").fused_attention(q, k, v, True, window=s["window"],
                                                 rope_theta=s["theta"])
    if kind == "attention32":
        q, k, v = s["qkv"]
        return _mod("fused_ops").fused_attention(q, k, v, s["causal"])
    if kind == "entropy":
        return s["plan"](s["logits"])
    if kind == "patches":
        P = _mod("patcher")
        mask, starts, lengths, counts = P.patch_boundaries(s["H"], PATCH_DELTA, out=s["out"])
        mH, mN, _ = P.patch_means(s["H"], s["N"], starts, counts, out=s["means"])
        return [mask, starts, lengths, counts, mH, mN]
    if kind == "row_ops":
        F = _mod("fused_ops")
        y = F.fused_rms_norm(s["x"], s["w"], 1e-5, l2_out=s["l2"])
        return [y, s["l2"], F.fused_silu_gate(s["a"], s["b"])]
    if kind == "pipeline":
        r = _mod("pipeline").process_document(s["data"], s["model"])
        return [r.entropies, r.norms,
                np.array([p.start_offset for p in r.patches], np.int64),
                np.array([p.length for p in r.patches], np.int64),
                np.array([p.prominence for p in r.patches], np.float32),
                np.array([p.entropy for p in r.patches], np.float32)]
    r = s["ingest"].run(s["tokens"], s["offsets"], patch_means=True)
    return [r.entropies, r.norms, r.coherence, r.starts, r.lengths, r.counts, r.patch_entropy,
            r.patch_prominence, r.patch_coherence]


# ---- what a pass cannot do without --------------------------------------------

def _pairs(T, window):
    w = min(window, T) if window > 0 else T
    return w * (w + 1) // 2 + (T - w) * w


def _layer_weights():
    return 4 * DIM * DIM + 3 * DIM * HIDDEN


def _chunks(n, chunk, overlap):
    """(start, end, kept from) of a document's chunks."""
    out, pos = [], 0
    while pos < n:
        start = max(0, pos - overlap) if pos else 0
        end = min(pos + chunk - overlap, n)
        out.append((start, end, pos - start))
        pos = end
    return out


def _pipeline_chunks(n):
    out, pos = [], 0
    while pos < n:
        end = min(pos + 4096, n)
        out.append((max(0, pos - 2048), end, pos - max(0, pos - 2048)))
        pos = end
    return out


def _model_flops(rows, window, layers, head=True):
    f = 0.0
    for T in rows:
        f += layers * (2.0 * T * _layer_weights() + 4.0 * 64 * HEADS * _pairs(T, window))
        f += 2.0 * T * DIM * VOCAB if head else 0.0
    return f


def work(case):
    kind = case["kind"]
    if kind in ("forward", "block"):
        layers, n = (LAYERS, case["batch"] * case["seq"]) if kind == "forward" else \
            (1, case["batch"] * case["seq"])
        head = kind == "forward"
        weights = 2.0 * layers * _layer_weights() + (2.0 * DIM * VOCAB if head else 0.0)
        out = n * 4.0 * (DIM + ((VOCAB + 3) if head else 0))
        return {"bytes": weights + 4.0 * n + out,
                "flops": _model_flops([case["seq"]] * case["batch"], case["window"], layers, head)}
    if kind == "attention":
        bh = case["batch"] * case["heads"]
        return {"bytes": 4.0 * bh * case["seq"] * 64 * 2,
                "flops": 4.0 * 64 * bh * _pairs(case["seq"], case["window"])}
    if kind == "attention32":
        bh, d, tq, tk = (case["batch"] * case["heads"], case["head_dim"], case["seq_q"],
                         case["seq_kv"])
        pairs = sum(min(i + 1, tk) for i in range(tq)) if case["causal"] else tq * tk
        return {"bytes": 4.0 * bh * d * (2 * tq + 2 * tk), "flops": 4.0 * d * bh * pairs}
    if kind == "entropy":
        n = case["batch"] * case["seq"]
        return {"bytes": n * (4.0 * case["vocab"] + 4 + 2 * 4), "flops": 5.0 * n * case["vocab"]}
    if kind == "patches":
        n = case["batch"] * case["seq"]
        return {"bytes": n * 12.0, "flops": 4.0 * n}
    if kind == "row_ops":
        e = 2 if case["dtype"] == "bf16" else 4
        n = case["rows"]
        return {"bytes": n * (2.0 * e * case["dim"] + 4 + 3.0 * e * case["hidden"]),
                "flops": n * (4.0 * case["dim"] + 6.0 * case["hidden"])}
    if kind == "pipeline":
        rows = [b - a for a, b, _ in _pipeline_chunks(case["bytes"])]
        return {"bytes": 2.0 * LAYERS * _layer_weights() + 9.0 * case["bytes"],
                "flops": _model_flops(rows, 512, LAYERS)}
    off = _doc_offsets(case)
    rows = [b - a for d in range(off.size - 1)
            for a, b, _ in _chunks(int(off[d + 1] - off[d]), case["chunk"], case["overlap"])]
    return {"bytes": 2.0 * LAYERS * _layer_weights() + 32.0 * float(off[-1]),
            "flops": _model_flops(rows, 512, LAYERS)}


# Four times the largest deviation of any output from exact() over the listed
# and drawn cases: bf16 operands with f32 accumulation in the model and the
# bf16 attention, bf16 results in the row ops, f32 elsewhere.
TOLERANCE = {
    "forward": {"rel": 2.2e-2},      # logits 5.8e-3
    "block": {"rel": 1.9e-2},        # 4.8e-3
    "attention": {"rel": 1.3e-2},    # 3.2e-3
    "attention32": {"rel": 3e-6},    # 8.1e-7 (d = 128, 1470 keys)
    "entropy": {"rel": 6e-7},        # 1.4e-7 (vocab 261)
    "pipeline": {"rel": 1.2e-3},     # norms 3.1e-4
    "ingest": {"rel": 2.8e-3},       # coherence 6.9e-4
}


def tolerance(case):
    kind = case["kind"]
    if kind == "patches":
        # the means are left-to-right f32 sums divided by the length, the
        # starts exact comparisons of the given f32 entropies
        return "exact"
    if kind == "row_ops":
        return {"rel": 7e-3 if case["dtype"] == "bf16" else 3e-7}  # 1.7e-3, 5.9e-8
    return TOLERANCE[kind]


# ---- 64-bit restatements --------------------------------------------------------

def _rope_table64(T, theta=10000.0):
    """The angles are f32 products by definition (pos * inv_freq in f32)."""
    inv = 1.0 / torch.tensor([theta ** (2 * i / 64) for i in range(32)], dtype=torch.float64
                             ).to(torch.float32)
    ang = (torch.arange(T, dtype=torch.float32)[:, None] * inv[None, :]).double()
    return ang.cos().to(DEV), ang.sin().to(DEV)


def _rotate64(x, cs, sn):
    a, b = x[..., :32], x[..., 32:]
    return torch.cat([a * cs - b * sn, a * sn + b * cs], -1)


def _attend64(q, k, v, causal, window):
    """[B, H, Tq, d] f64; keys j <= i (causal), j > i - window (window > 0)."""
    Tq, Tk, d = q.shape[2], k.shape[2], q.shape[3]
    out = torch.empty_like(q)
    step = 256
    for i0 in range(0, Tq, step):
        i1 = min(i0 + step, Tq)
        lo = max(0, i0 - window + 1) if causal and window > 0 else 0
        hi = min(Tk, i1) if causal else Tk
        kk = k[:, :, lo:hi].transpose(2, 3).contiguous()
        s = torch.matmul(q[:, :, i0:i1].contiguous(), kk) / math.sqrt(d)
        if causal:
            i = torch.arange(i0, i1, device=DEV)[:, None]
            j = torch.arange(lo, hi, device=DEV)[None, :]
            ok = j <= i
            if window > 0:
                ok &= j > i - window
            s = s.masked_fill(~ok, -math.inf)
        out[:, :, i0:i1] = torch.matmul(torch.softmax(s, -1), v[:, :, lo:hi].contiguous())
    return out


_weights64 = {}


def _device_weights(layers):
    """The bf16 weights on the device (converted to f64 a layer at a time)."""
    if layers not in _weights64:
        _weights64[layers] = {
            n: torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).to(DEV).view(torch.bfloat16)
            for n, a in _get_weights(layers)[1].items()}
    return _weights64[layers]


def _rms64(x, w):
    return x / (x.pow(2).mean(-1, keepdim=True).sqrt() + 1e-5) * w


def _forward64(tokens, window, layers, head=True):
    """Tokens [T] -> (residual, logits, norms, entropies, coherence) in f64."""
    w = _device_weights(layers)
    x = w["tok_embeddings"].double()[tokens.long()]
    T = x.shape[0]
    cs, sn = _rope_table64(T)
    heads = lambda t: t.view(1, T, HEADS, 64).transpose(1, 2)  # noqa: E731
    for l in range(layers):
        g = lambda n: w[n][l].double()  # noqa: E731
        h = _rms64(x, g("attention_norm"))
        q = _rotate64(heads(h @ g("wq")), cs, sn)
        k = _rotate64(heads(h @ g("wk")), cs, sn)
        a = _attend64(q, k, heads(h @ g("wv")), True, window)
        x = x + a.transpose(1, 2).reshape(T, DIM) @ g("wo")
        h = _rms64(x, g("ffn_norm"))
        x = x + (torch.nn.functional.silu(h @ g("w1")) * (h @ g("w3"))) @ g("w2")
    if not head:
        return x
    norms = x.norm(dim=-1)
    logits = _rms64(x, w["norm"].double()) @ w["output"].double()
    H = _entropy64(logits)
    return x, logits, norms, H, norms * norms / (H + 1e-6)


def _chunked64(tokens, chunks):
    parts = []
    for a, b, skip in chunks:
        t = torch.from_numpy(np.ascontiguousarray(tokens[a:b])).to(DEV)
        _, _, n, H, c = _forward64(t, 512, LAYERS)
        parts.append([y[skip:] for y in (H, n, c)])
    return [torch.cat(p).cpu().numpy() for p in zip(*parts)]


def exact(case, seed):
    kind = case["kind"]
    if kind == "forward":
        tok = torch.from_numpy(_tokens(case, seed)).to(DEV)
        rows = [_forward64(t, case["window"], LAYERS) for t in tok]
        x, lg, n, H, c = (torch.stack(p) for p in zip(*rows))
        return [lg, x, n, H, c]
    if kind == "block":
        tok = torch.from_numpy(_tokens(case, seed)).to(DEV)
        return torch.stack([_forward64(t, case["window"], 1, head=False) for t in tok])
    if kind == "attention":
        q, k, v = (t.double() for t in _attention_inputs(case, seed))
        if case["theta"] > 0:
            cs, sn = _rope_table64(case["seq"], case["theta"])
            q, k = _rotate64(q, cs, sn), _rotate64(k, cs, sn)
        return _attend64(q, k, v, True, case["window"])
    if kind == "attention32":
        q, k, v = (t.double() for t in _attention32_inputs(case, seed))
        return _attend64(q, k, v, case["causal"], 0)
    if kind == "entropy":
        H = _entropy64(_logits(case, seed))
        return [H, [_starts64(H, mode, thr) for mode, thr in ENTROPY_RULES]]
    if kind == "patches":
        H, N = _signals(case, seed)
        mask, starts, lengths, counts = _starts64(H, 0, PATCH_DELTA)
        means = []
        for x in (H.double().cpu().numpy(), N.double().cpu().numpy()):
            m = np.zeros(x.shape)
            for b in range(x.shape[0]):
                n = int(counts[b])
                m[b, :n] = np.add.reduceat(x[b], starts[b, :n]) / lengths[b, :n]
            means.append(m)
        return [mask, starts, lengths, counts] + means
    if kind == "row_ops":
        x, w, a, b = (t.double() for t in _row_inputs(case, seed))
        return [_rms64(x, w), x.norm(dim=-1), torch.nn.functional.silu(a) * b]
    if kind == "pipeline":
        data = _document(case, seed).astype(np.int32)
        H, n, _ = _chunked64(data, _pipeline_chunks(data.size))
        return [H, n, None, None, None, None]
    tok, off = _documents(case, seed)
    docs = [_chunked64(tok[off[d]:off[d + 1]], _chunks(int(off[d + 1] - off[d]), case["chunk"],
                                                        case["overlap"]))
            for d in range(off.size - 1)]
    return [np.concatenate(p) for p in zip(*docs)] + [None] * 6


def _starts64(H, mode, thr):
    """Mask, starts, lengths and counts of one boundary rule (patches are
    decided on the f32 entropies' f32 differences)."""
    h = H.float().cpu().numpy()
    B, T = h.shape
    mask = np.zeros((B, T), np.int32)
    mask[:, :2] = 1
    if T > 2:
        step = h[:, 2:] - h[:, 1:-1] if mode == 0 else h[:, 2:]
        mask[:, 2:] = step > np.float32(thr)
    starts, lengths = np.zeros((B, T), np.int32), np.zeros((B, T), np.int32)
    counts = mask.sum(1).astype(np.int32)
    for b in range(B):
        s = np.flatnonzero(mask[b])
        starts[b, :s.size] = s
        lengths[b, :s.size] = np.diff(np.append(s, T))
    return [mask, starts, lengths, counts]
