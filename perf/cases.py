"""The work a transcription program has this framework do, as cases that can be timed.

One case per stage of the pipeline, at large-v3 width (20 heads of 64, vocabulary 51866, 448 text
positions, 1500 encoder rows): audio to log-mel, encoder self-attention, the prompt's and the draft's
cached attention, whole decode steps, greedy sampling, and the word alignment's uncached attention
and score preparation. ``listed`` gives fixed cases, ``draw`` random ones of the same ranges.
``prepare`` makes what the program holds before the call, ``run`` is one pass through the public
entry points, ``exact`` the same result in 64-bit torch.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

D = 64
VOCAB = 51866
SELF_LEN = 448
CROSS_LEN = 1500
BUCKETS = [1, 2, 4, 8, 16, 32, 42, 52, 54]
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # one 30-s window of a live stream through the front end (latency: three small launches)
        {"name": "mel_window", "kind": "mel", "batch": 1, "samples": 480000, "mels": 128, "frames": 3000},
        # a file cut into 16 windows, all at once
        {"name": "mel_batch", "kind": "mel", "batch": 16, "samples": 480000, "mels": 128, "frames": 3000},
        # one encoder layer's attention for one window (fp16 checkpoints): fewer blocks than CUs
        {"name": "encoder_window", "kind": "encoder", "dtype": "fp16", "batch": 1, "heads": 20, "length": 1500},
        # the same for a batch of 16 windows, the framework's throughput shape
        {"name": "encoder_batch", "kind": "encoder", "dtype": "bf16", "batch": 16, "heads": 20, "length": 1500},
        # full-precision encoder layer (the reference configuration results are checked with)
        {"name": "encoder_fp32", "kind": "encoder", "dtype": "fp32", "batch": 1, "heads": 20, "length": 1500},
        # the previous text as prompt: 16 streams append 224 tokens and attend, self then cross
        {"name": "prompt", "kind": "cached", "dtype": "bf16", "streams": 16, "tokens": 224, "heads": 20, "filled": 0},
        # speculative decoding: 16 streams verify a 5-token draft behind ragged histories
        {"name": "verify", "kind": "cached", "dtype": "fp16", "streams": 16, "tokens": 5, "heads": 20, "filled": 400},
        # one token of a single live stream: a whole captured decode step of four layers
        {"name": "step_one", "kind": "step", "dtype": "bf16", "streams": 1, "layers": 4, "heads": 20},
        # one token of 52 streams, the reference's default slot count
        {"name": "step_batch", "kind": "step", "dtype": "bf16", "streams": 52, "layers": 4, "heads": 20},
        # the sampling tail after that step: masks, repetition penalty, greedy token
        {"name": "sample", "kind": "sample", "dtype": "bf16", "rows": 52, "vocab": VOCAB},
        # word alignment re-runs the text uncached: causal self and cross attention of one layer
        {"name": "text", "kind": "text", "dtype": "bf16", "batch": 16, "heads": 20, "length": 448, "audio": 1500},
        # ... and turns the ten alignment heads' projections into the matrix the path search takes
        {"name": "align", "kind": "align", "dtype": "bf16", "batch": 16, "heads": 10, "length": 448, "audio": 1500},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["mel", "encoder", "cached", "step", "sample", "text", "align"])
    low = rng.choice(["bf16", "fp16"])
    if kind == "mel":
        n = rng.choice([480000, rng.randint(16000, 480000)])
        return {"kind": kind, "batch": _log(rng, 1, 16), "samples": n, "mels": rng.choice([80, 128]),
                "frames": rng.choice([3000, n // 160])}
    if kind == "encoder":
        dtype = rng.choice(["bf16", "fp16", "bf16", "fp16", "fp32"])
        return {"kind": kind, "dtype": dtype, "batch": _log(rng, 1, 2 if dtype == "fp32" else 16),
                "heads": rng.choice([6, 8, 12, 16, 20]), "length": rng.choice([1500, rng.randint(300, 1500)])}
    if kind == "cached":
        return {"kind": kind, "dtype": low, "streams": _log(rng, 1, 64), "tokens": _log(rng, 1, 224),
                "heads": rng.choice([6, 12, 20]), "filled": rng.choice([0, rng.randint(1, 220)])}
    if kind == "step":
        return {"kind": kind, "dtype": low, "streams": _log(rng, 1, 52), "layers": 4, "heads": rng.choice([8, 12, 20])}
    if kind == "sample":
        return {"kind": kind, "dtype": rng.choice(["bf16", "fp16", "fp32"]), "rows": _log(rng, 1, 64),
                "vocab": rng.choice([51864, 51865, VOCAB])}
    if kind == "text":
        return {"kind": kind, "dtype": low, "batch": _log(rng, 1, 16), "heads": rng.choice([6, 12, 20]),
                "length": rng.randint(20, 448), "audio": rng.choice([1500, rng.randint(200, 1500)])}
    return {"kind": kind, "dtype": low, "batch": _log(rng, 1, 16), "heads": rng.randint(4, 10),
            "length": rng.randint(20, 448), "audio": rng.choice([1500, rng.randint(300, 1500)])}


# ---- inputs -----------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _host(seed):
    import random

    return random.Random(seed)


def _randn(g, *shape, dtype=torch.float32, std=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * std).to(dtype)


def _lengths(seed, n, lo, hi):
    """Ragged lengths of n rows."""
    r = _host(seed)
    return [r.randint(lo, hi) for _ in range(n)]


def _mel_audio(case, seed):
    """Speech-like audio: noise and a few tones under a slow envelope, with a silent stretch."""
    g = _gen(seed)
    B, N = case["batch"], case["samples"]
    t = torch.arange(N, device="cuda", dtype=torch.float32) / 16000.0
    f = 100.0 + 3000.0 * torch.rand((B, 4), generator=g, device="cuda")
    x = 0.02 * torch.randn((B, N), generator=g, device="cuda")
    for i in range(4):
        x += 0.1 * torch.sin(2 * math.pi * f[:, i : i + 1] * t)
    x *= 0.5 + 0.5 * torch.sin(2 * math.pi * 1.3 * t)
    x[:, N // 3 : N // 3 + N // 20] = 0.0
    return x


def _heads_view(x, heads):
    B, T, _ = x.shape
    return x.view(B, T, heads, D).permute(0, 2, 1, 3)


def _histories(case, seed):
    """Tokens already cached per stream: none, or ragged up to ``filled``."""
    if not case["filled"]:
        return [0] * case["streams"]
    return _lengths(seed, case["streams"], 1, min(case["filled"], SELF_LEN - case["tokens"]))


def _cached_inputs(case, seed):
    g = _gen(seed)
    dt, B, T, H = DTYPES[case["dtype"]], case["streams"], case["tokens"], case["heads"]
    st = {n: _randn(g, B, T, H, D, dtype=dt) for n in ("q", "k", "v", "qx")}
    for n, rows in (("ks", SELF_LEN), ("vs", SELF_LEN), ("kx", CROSS_LEN), ("vx", CROSS_LEN)):
        # head-major storage seen as [slot, position, head, dim], as the slot caches keep it
        st[n] = _randn(g, B, H, rows, D, dtype=dt).permute(0, 2, 1, 3)
    st["cs"] = torch.tensor(_histories(case, seed), dtype=torch.int32, device="cuda")
    slots = list(range(B))
    _host(seed + 1).shuffle(slots)
    st["slots"] = torch.tensor(slots, dtype=torch.int32, device="cuda")
    return st


def _bucket(streams):
    return next(b for b in BUCKETS if streams <= b)


def _step_weights(case, seed):
    """A decoder's parameters by name, scaled so that every layer moves the residual stream."""
    g, dt, n = _gen(seed), DTYPES[case["dtype"]], case["heads"] * D
    w = {"token_embedding.weight": _randn(g, VOCAB, n, dtype=dt, std=0.05),
         "positional_embedding": _randn(g, SELF_LEN, n, dtype=dt, std=0.02)}

    def norm(name):
        w[name + ".weight"] = (1 + _randn(g, n, std=0.1)).to(dt)
        w[name + ".bias"] = _randn(g, n, dtype=dt, std=0.1)

    def linear(name, rows, cols, bias=True):
        w[name + ".weight"] = _randn(g, rows, cols, dtype=dt, std=cols ** -0.5)
        if bias:
            w[name + ".bias"] = _randn(g, rows, dtype=dt, std=0.1)

    for i in range(case["layers"]):
        for part in ("attn", "cross_attn"):
            norm(f"blocks.{i}.{part}_ln")
            for m in ("query", "key", "value", "out"):
                linear(f"blocks.{i}.{part}.{m}", n, n, bias=m != "key")
        norm(f"blocks.{i}.mlp_ln")
        linear(f"blocks.{i}.mlp.0", 4 * n, n)
        linear(f"blocks.{i}.mlp.2", n, 4 * n)
    norm("ln")
    return w


def _step_lengths(case, seed):
    """Ragged histories of the streams; the bucket's padding rows keep one token."""
    return _lengths(seed, case["streams"], 1, 400) + [1] * (_bucket(case["streams"]) - case["streams"])


def _step_tokens(case, seed):
    return torch.randint(0, VOCAB, (case["streams"], 1), generator=_gen(seed + 1), device="cuda")


def _step_caches(case, seed, layer):
    """One layer's self and cross K/V, head-major: [slots, heads, rows, head_dim]."""
    g, dt, n, H = _gen(seed + 2 + layer), DTYPES[case["dtype"]], _bucket(case["streams"]), case["heads"]
    return [_randn(g, n, H, rows, D, dtype=dt) for rows in (SELF_LEN, SELF_LEN, CROSS_LEN, CROSS_LEN)]


def _step_state(case, seed):
    from whisperdrz_amd.decoder import BucketedDecodeGraphs, TextDecoderStack
    from whisperdrz_amd.kv_cache import KVSlotPool

    dt, H, L, n = DTYPES[case["dtype"]], case["heads"], case["layers"], _bucket(case["streams"])
    with torch.device("meta"):
        dec = TextDecoderStack(VOCAB, SELF_LEN, H * D, H, L)
    dec.load_state_dict(_step_weights(case, seed), assign=True)
    dec = dec.to(dt).eval()
    pool = KVSlotPool(L, n, H, D, self_len=SELF_LEN, cross_len=CROSS_LEN, dtype=dt, device="cuda")
    graphs = BucketedDecodeGraphs(dec, pool, VOCAB, buckets=[n])
    with torch.no_grad():
        graphs.capture(n)
    for i, (s, c) in enumerate(zip(pool.self_kv, pool.cross_kv)):
        for storage, rows in zip((s.k_storage, s.v_storage, c.k_storage, c.v_storage), _step_caches(case, seed, i)):
            storage.copy_(rows)
    lens = torch.tensor(_step_lengths(case, seed), dtype=torch.int32, device="cuda")
    B = case["streams"]
    return {"graphs": graphs, "pool": pool, "lens": lens.expand(L, n).contiguous(), "tokens": _step_tokens(case, seed),
            "positions": lens[:B].long(), "slots": torch.arange(B, device="cuda")}


def _align_inputs(case, seed):
    """Captured projections of five layers, with the alignment heads spread over them."""
    g = _gen(seed)
    dt, B, T, A, width = DTYPES[case["dtype"]], case["batch"], case["length"], case["audio"], 20
    mask = torch.zeros(5, width, dtype=torch.bool)
    for i in range(case["heads"]):
        mask[i % 5, (7 * i) % width] = True
    q = [_randn(g, B, T, width * D, dtype=dt) for _ in range(5)]
    k = [_randn(g, B, A, width * D, dtype=dt) for _ in range(5)]
    lens = _lengths(seed, B, max(1, T // 2), T)
    caps = _lengths(seed + 1, B, max(1, A // 2), A)
    caps[0] = A
    return q, k, mask, lens, caps


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mel":
        from whisperdrz_amd import LogMelSpectrogram

        return {"case": case, "audio": _mel_audio(case, seed), "front": LogMelSpectrogram(case["mels"])}
    if kind == "encoder":
        g = _gen(seed)
        shape = (case["batch"], case["length"], case["heads"] * D)
        return {"case": case, "qkv": [_randn(g, *shape, dtype=DTYPES[case["dtype"]]) for _ in range(3)]}
    if kind == "cached":
        return {"case": case, **_cached_inputs(case, seed)}
    if kind == "step":
        return {"case": case, **_step_state(case, seed)}
    if kind == "sample":
        g = _gen(seed)
        rows, V = case["rows"], case["vocab"]
        rand = torch.rand((2, rows, VOCAB), generator=g, device="cuda")
        return {"case": case, "logits": _randn(g, rows, V, dtype=DTYPES[case["dtype"]], std=4.0),
                "blocked": (rand[0] < 0.03), "penalty": (rand[1] < 0.002)}
    if kind == "text":
        g = _gen(seed)
        dt, B, n = DTYPES[case["dtype"]], case["batch"], case["heads"] * D
        return {"case": case, "self": [_randn(g, B, case["length"], n, dtype=dt) for _ in range(4)],
                "cross": [_randn(g, B, case["audio"], n, dtype=dt) for _ in range(2)]}
    return {"case": case, "inputs": _align_inputs(case, seed)}


# ---- one pass ---------------------------------------------------------------------------------


def run(state):
    import whisperdrz_amd as wd

    case = state["case"]
    kind = case["kind"]
    if kind == "mel":
        return state["front"](state["audio"], target_frames=case["frames"])
    if kind == "encoder":
        q, k, v = state["qkv"]
        return wd.qkv_attention(q, k, v, case["heads"])
    if kind == "cached":
        o = wd.flash_attn_with_kvcache(state["q"], state["ks"], state["vs"], k=state["k"], v=state["v"],
                                       cache_seqlens=state["cs"], cache_batch_idx=state["slots"],
                                       softmax_scale=D ** -0.5, causal=True)
        x = wd.flash_attn_with_kvcache(state["qx"], state["kx"], state["vx"], cache_batch_idx=state["slots"],
                                       softmax_scale=D ** -0.5)
        return {"self": o, "cross": x, "k_cache": state["ks"], "v_cache": state["vs"]}
    if kind == "step":
        # the lengths as they stand before this token: a pass appends at the same positions each time
        state["pool"].self_seq_lens.copy_(state["lens"])
        with torch.no_grad():
            logits = state["graphs"].forward(state["tokens"], state["positions"], state["slots"])
        rows = [c[: case["streams"]] for s in state["pool"].self_kv for c in (s.k_cache, s.v_cache)]
        return {"logits": logits, "lengths": state["pool"].self_seq_lens, "caches": rows}
    if kind == "sample":
        return wd.masked_argmax(state["logits"], state["blocked"], state["penalty"])
    if kind == "text":
        q, k, v, qx = state["self"]
        kx, vx = state["cross"]
        return {"self": wd.qkv_attention(q, k, v, case["heads"], causal=True),
                "cross": wd.qkv_attention(qx, kx, vx, case["heads"])}
    q, k, mask, lens, caps = state["inputs"]
    return wd.dtw_attention_prep(q, k, mask, lens, caps)


# ---- what a pass cannot do without --------------------------------------------------------------


def work(case):
    kind = case["kind"]
    e = 4 if case.get("dtype") == "fp32" else 2
    if kind == "mel":
        B, n = case["batch"], case["samples"] // 160
        # a real 400-point FFT per frame (2.5 N log2 N), powers, and the two-band filterbank
        flops = B * n * (2.5 * 400 * math.log2(400) + 3 * 201 + 4 * 201)
        return {"bytes": 4 * B * (case["samples"] + case["mels"] * case["frames"]), "flops": flops}
    if kind == "encoder":
        B, H, L = case["batch"], case["heads"], case["length"]
        return {"bytes": 4 * B * H * L * D * e, "flops": 4 * B * H * L * L * D}
    if kind == "cached":
        B, H, T = case["streams"], case["heads"], case["tokens"]
        hist = case["filled"] // 2
        row = B * H * D * e
        keys = B * H * (T * hist + T * (T + 1) / 2 + T * CROSS_LEN)
        # q, k, v, qx read, two outputs and the appended rows written, the caches' valid rows read
        return {"bytes": row * (4 * T + 2 * T + 2 * T + 2 * hist + 2 * CROSS_LEN), "flops": 4 * D * keys}
    if kind == "step":
        B, H, L = case["streams"], case["heads"], case["layers"]
        n = H * D
        weights = L * 14 * n * n + VOCAB * n
        kv = L * B * 2 * n * (200 + CROSS_LEN)
        return {"bytes": e * (weights + kv + B * VOCAB), "flops": 2 * B * weights + 2 * kv}
    if kind == "sample":
        return {"bytes": case["rows"] * case["vocab"] * (e + 2) + 8 * case["rows"], "flops": 3 * case["rows"] * case["vocab"]}
    if kind == "text":
        B, H, T, A = case["batch"], case["heads"], case["length"], case["audio"]
        return {"bytes": B * H * D * e * (4 * T + 2 * T + 2 * A),
                "flops": 4 * B * H * D * (T * (T + 1) / 2 + T * A)}
    B, H, T, A = case["batch"], case["heads"], case["length"], case["audio"]
    return {"bytes": B * H * (T + A) * D * e + 4 * B * T * A, "flops": B * H * T * A * (2 * D + 20)}


def tolerance(case):
    """About four times the distance from 64 bits that the rounding of the types gives."""
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "mel":
        return {"rel": 4e-6}
    if kind == "align":
        return {"rel": 2e-6}
    if kind == "step":
        return {"rel": 3.5e-2 if case["dtype"] == "bf16" else 4e-3}
    return {"rel": {"bf16": 1e-2, "fp16": 1.5e-3, "fp32": 2e-6}[case["dtype"]]}


# ---- the same in 64 bits --------------------------------------------------------------------------


def _attend(q, k, v, scale, hidden=None):
    """softmax(q k^T scale) v over [..., L, D] in 64 bits; ``hidden`` masks keys."""
    s = q.double() @ k.double().transpose(-1, -2) * scale
    if hidden is not None:
        s = s.masked_fill(hidden, -math.inf)
    return torch.softmax(s, -1) @ v.double()


def _sdpa(q, k, v, heads, causal):
    """Per batch row, so that the scores of a large batch fit."""
    hidden = None
    if causal:
        i = torch.arange(q.shape[1], device=q.device)
        hidden = i[None, :] > i[:, None]
    out = []
    for b in range(q.shape[0]):
        o = _attend(*(_heads_view(t[b : b + 1], heads) for t in (q, k, v)), D ** -0.5, hidden)
        out.append(o.permute(0, 2, 1, 3).reshape(1, q.shape[1], -1))
    return torch.cat(out)


def _mel_filters(n_mels):
    """The slaney filterbank, [201, n_mels] in 64 bits."""
    f_sp, logstep = 200.0 / 3.0, math.log(6.4) / 27.0
    top = 1000.0 / f_sp + math.log(8.0) / logstep
    mels = torch.linspace(0.0, top, n_mels + 2, dtype=torch.float64)
    hz = torch.where(mels < 15.0, mels * f_sp, 1000.0 * torch.exp(logstep * (mels - 15.0)))
    bins = torch.linspace(0.0, 8000.0, 201, dtype=torch.float64)
    down = (bins[:, None] - hz[None, :-2]) / (hz[1:-1] - hz[:-2])
    up = (hz[None, 2:] - bins[:, None]) / (hz[2:] - hz[1:-1])
    return torch.clamp(torch.minimum(down, up), min=0.0) * (2.0 / (hz[2:] - hz[:-2]))


def _mel_exact(case, seed):
    out = []
    fb = _mel_filters(case["mels"]).cuda()
    window = torch.hann_window(400, dtype=torch.float64, device="cuda")
    for x in _mel_audio(case, seed).double():
        spec = torch.stft(x, 400, 160, window=window, center=True, pad_mode="reflect", return_complex=True)
        mel = fb.T @ spec[:, :-1].abs().square()
        lg = torch.log10(torch.clamp(mel, min=1e-10))
        lg = (torch.maximum(lg, lg.max() - 8.0) + 4.0) / 4.0
        n = case["frames"]
        out.append(lg[:, :n] if lg.shape[1] >= n else F.pad(lg, (0, n - lg.shape[1]), value=-1.5))
    return torch.stack(out)


def _cached_exact(case, seed):
    st = _cached_inputs(case, seed)
    T, scale = case["tokens"], D ** -0.5
    o, x = [], []
    for b, (cs, slot) in enumerate(zip(st["cs"].tolist(), st["slots"].tolist())):
        st["ks"][slot, cs : cs + T] = st["k"][b]
        st["vs"][slot, cs : cs + T] = st["v"][b]
        j, t = torch.arange(cs + T, device="cuda"), torch.arange(T, device="cuda")
        per_head = lambda a: a.transpose(0, 1)
        ks, vs = per_head(st["ks"][slot, : cs + T]), per_head(st["vs"][slot, : cs + T])
        o.append(per_head(_attend(per_head(st["q"][b]), ks, vs, scale, j[None, :] > cs + t[:, None])))
        x.append(per_head(_attend(per_head(st["qx"][b]), per_head(st["kx"][slot]), per_head(st["vx"][slot]), scale)))
    return {"self": torch.stack(o), "cross": torch.stack(x), "k_cache": st["ks"].double(), "v_cache": st["vs"].double()}


def _step_exact(case, seed):
    B, H = case["streams"], case["heads"]
    w = {name: p.double() for name, p in _step_weights(case, seed).items()}
    lens = _step_lengths(case, seed)[:B]
    lin = lambda name, x: F.linear(x, w[name + ".weight"], w.get(name + ".bias"))
    norm = lambda name, x: F.layer_norm(x, (H * D,), w[name + ".weight"], w[name + ".bias"], 1e-5)
    caches = []
    x = w["token_embedding.weight"][_step_tokens(case, seed)[:, 0]] + w["positional_embedding"][lens]
    for i in range(case["layers"]):
        p = f"blocks.{i}."
        sk, sv, ck, cv = _step_caches(case, seed, i)
        h = norm(p + "attn_ln", x)
        q, k, v = (lin(f"{p}attn.{m}", h).view(B, H, 1, D) for m in ("query", "key", "value"))
        sk, sv = sk[:B].double(), sv[:B].double()
        for b, n in enumerate(lens):
            sk[b, :, n], sv[b, :, n] = k[b, :, 0], v[b, :, 0]
        caches += [sk.permute(0, 2, 1, 3), sv.permute(0, 2, 1, 3)]
        o = [_attend(q[b], sk[b, :, : n + 1], sv[b, :, : n + 1], D ** -0.5) for b, n in enumerate(lens)]
        x = x + lin(p + "attn.out", torch.stack(o).reshape(B, H * D))
        q = lin(p + "cross_attn.query", norm(p + "cross_attn_ln", x)).view(B, H, 1, D)
        o = [_attend(q[b], ck[b], cv[b], D ** -0.5) for b in range(B)]
        x = x + lin(p + "cross_attn.out", torch.stack(o).reshape(B, H * D))
        x = x + lin(p + "mlp.2", F.gelu(lin(p + "mlp.0", norm(p + "mlp_ln", x))))
    logits = norm("ln", x) @ w["token_embedding.weight"].T
    return {"logits": logits.view(B, 1, VOCAB), "lengths": None, "caches": caches}


def _align_exact(case, seed):
    q, k, mask, lens, caps = _align_inputs(case, seed)
    T, A, C = case["length"], case["audio"], max(caps)
    out = []
    for b, (n, cap) in enumerate(zip(lens, caps)):
        total = 0.0
        for layer, head in mask.nonzero().tolist():
            cols = slice(head * D, (head + 1) * D)
            s = q[layer][b, :, cols].double() @ k[layer][b, :, cols].double().T * D ** -0.5
            s[:, cap:] = -math.inf
            w = torch.softmax(s, -1)
            std, mean = torch.std_mean(w[:n], dim=0, unbiased=False)
            w = (w - mean) / std.clamp_min(1e-6)
            w = F.pad(w[None], (3, 3), mode="reflect")[0].unfold(-1, 7, 1)
            total = total + w.median(-1).values
        out.append((total / mask.sum())[:, :C])
    return torch.stack(out)


def exact(case, seed):
    kind = case["kind"]
    if kind == "mel":
        return _mel_exact(case, seed)
    if kind == "encoder":
        q, k, v = prepare(case, seed)["qkv"]
        return _sdpa(q, k, v, case["heads"], False)
    if kind == "cached":
        return _cached_exact(case, seed)
    if kind == "step":
        return _step_exact(case, seed)
    if kind == "text":
        st = prepare(case, seed)
        q, k, v, qx = st["self"]
        return {"self": _sdpa(q, k, v, case["heads"], True), "cross": _sdpa(qx, *st["cross"], case["heads"], False)}
    if kind == "align":
        return _align_exact(case, seed)
    return None  # sampled tokens are picked, not computed
