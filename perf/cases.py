"""The workloads whose speed is tracked: what a program built on this package runs.

Five families, each through the public entry points:

* ``linear``  one projection, ``QMatMul.forward`` (the drop-in for Candle's QMatMul): any
  weight format, row count, bias, f32 or bf16 input;
* ``prompt``  prompt prefill of an engine (ragged streams);
* ``decode``  autoregressive steps of an engine whose streams hold a prompt, restarted from
  that prompt on every pass (a server that keeps a voice prompt cached and rewinds to it);
* ``frame``   Fish dual-AR frames: slow step, semantic draw, fast-AR expansion;
* ``load``    weight ingest: ``QTensor.quantize`` of an f32 matrix.

Steps and frames are fed given tokens (the drawn ones are outputs), so every pass does the
same work and the outputs of two builds can be compared position by position.  Weights are
normal and encoded here into GGML blocks, as a GGUF file brings them; activations and
embeddings are N(0, 1).  ``exact`` states the same computation in plain torch, 64-bit.
"""
from __future__ import annotations

import math

import torch

from syrinx_amd.decoder import (ATTN_NORM, BK, BQ, BV, CODEBOOK_EMBED, EMBED, FFN_NORM, FINAL_NORM, HEAD, HEAD_BIAS,
                                K_NORM, Q_NORM, W1, W2, W3, WO, WQKV, DecoderLM, FastAr, Qwen2Lm, SlowAr,
                                cosyvoice2_lm_config, fish_s2_fast_ar_config, fish_s2_slow_ar_config)
from syrinx_amd.quantized import GgmlDType, QMatMul, QTensor
from syrinx_amd.sampling import FishSampler, RasSampler, SamplingParams

DEV = "cuda:0"
F64 = torch.float64
BLOCK = {"q4k": 256, "q8_0": 32, "q4_0": 32}
BLOCK_BYTES = {"q4k": 144, "q8_0": 34, "q4_0": 18}
DTYPE = {"q4k": GgmlDType.Q4K, "q8_0": GgmlDType.Q8_0, "q4_0": GgmlDType.Q4_0}


# ---- the cases ------------------------------------------------------------------------

def listed():
    return [
        # one token through the smallest projection of the CosyVoice2 LM (k_proj with its
        # bias): latency and launches only
        _linear("linear_q8_0_1x896x128", "q8_0", 128, 896, 1, True, False),
        # a short sentence's rows through the CosyVoice2 MLP up-projection
        _linear("linear_q8_0_50x896x4864", "q8_0", 4864, 896, 50, False, False),
        # a short Fish prompt, bf16 activations as the reference's GPU path keeps them
        _linear("linear_q4k_37x2560x6144_bf16", "q4k", 6144, 2560, 37, False, True),
        # the CosyVoice3 flow's DiT feed-forward: 2 x 250 frames
        _linear("linear_q4_0_500x1024x2048", "q4_0", 2048, 1024, 500, True, False),
        # many prompts' rows at once through the widest Fish projection (gate|up)
        _linear("linear_q4k_2048x2560x19456", "q4k", 19456, 2560, 2048, False, False),
        # ragged prompts of three requests through four layers of the Fish block
        {"name": "prompt_fish_ragged", "family": "prompt", "model": "fish", "layers": 4, "counts": "311,1024,77",
         "all": False},
        # the CosyVoice2 LM over an utterance's step-0 input, logits of every position
        {"name": "prompt_cv2_226", "family": "prompt", "model": "cv2", "layers": 24, "counts": "226", "all": True},
        # one Fish utterance: whole frames of the full model
        {"name": "frame_fish_1", "family": "frame", "lens": "640", "frames": 4},
        # 16 concurrent streams with ragged caches through four layers of the Fish block
        {"name": "decode_fish_16", "family": "decode", "model": "fish", "layers": 4, "steps": 4,
         "lens": "1203,414,1845,980,256,1677,733,2040,1390,577,1121,1958,301,861,1544,1099"},
        # one CosyVoice2 utterance, token by token with the RAS draw
        {"name": "decode_cv2_1", "family": "decode", "model": "cv2", "layers": 24, "steps": 16, "lens": "500"},
        # eight concurrent CosyVoice2 utterances
        {"name": "decode_cv2_8", "family": "decode", "model": "cv2", "layers": 24, "steps": 8,
         "lens": "226,511,389,602,97,450,318,275"},
        # a checkpoint's w2 cast to Q4_K at load
        {"name": "load_q4k_2560x9728", "family": "load", "dtype": "q4k", "n": 2560, "k": 9728},
    ]


def _linear(name, dtype, n, k, m, bias, bf16):
    return {"name": name, "family": "linear", "dtype": dtype, "n": n, "k": k, "m": m, "bias": bias, "bf16": bf16}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["linear", "linear", "linear", "prompt", "decode", "decode", "frame", "load"])
    if family in ("linear", "load"):
        dtype = rng.choice(["q4k", "q8_0", "q4_0"])
        bs = BLOCK[dtype]
        n, k = _log(rng, 80, 19456), max(1, _log(rng, 256, 9728) // bs) * bs
        if family == "load":
            return {"family": family, "dtype": dtype, "n": n, "k": k}
        while n * k > 19456 * 2560:
            n = n // 2 + 1
        case = _linear("", dtype, n, k, _log(rng, 1, 2048), rng.random() < 0.5, rng.random() < 0.3)
        del case["name"]
        return case
    if family == "frame":
        lens = ",".join(str(_log(rng, 16, 1024)) for _ in range(rng.randint(1, 3)))
        return {"family": family, "lens": lens, "frames": 2}
    model = rng.choice(["fish", "cv2"])
    if family == "prompt":
        n, total = rng.randint(1, 4), 1400 if model == "fish" else 700
        counts = ",".join(str(_log(rng, 1, total // n)) for _ in range(n))
        return {"family": family, "model": model, "layers": rng.randint(2, 4) if model == "fish" else 24,
                "counts": counts, "all": model == "cv2"}
    n = _log(rng, 1, 16)
    lens = ",".join(str(_log(rng, 16, 2000 if model == "fish" else 900)) for _ in range(n))
    return {"family": family, "model": model, "layers": rng.randint(2, 4) if model == "fish" else 24, "steps": 4,
            "lens": lens}


def _ints(text):
    return [int(v) for v in text.split(",")]


# ---- seeded data ----------------------------------------------------------------------

def _gen(seed, *path):
    s = seed & 0xFFFFFFFF
    for p in path:
        s = (s * 1000003 + p + 1) & 0x7FFFFFFFFFFF
    return torch.Generator(device=DEV).manual_seed(s)


def _normal(shape, std, seed, *path):
    return torch.randn(shape, generator=_gen(seed, *path), device=DEV).mul_(std)


def _round(x):
    return torch.floor(x + 0.5)


def _encode(dtype, w):
    """f32 [n, k] -> (GGML blocks uint8 [n, bytes], the parameters of the decoded weight)."""
    n, k = w.shape
    b = w.view(n, k // BLOCK[dtype], BLOCK[dtype])
    if dtype != "q4k":
        amax = b.abs().amax(-1, keepdim=True)
        d = (amax / (127 if dtype == "q8_0" else 8)).half()
        q = _round(b / d.float().clamp_min(1e-30))
        if dtype == "q8_0":
            q = q.clamp_(-127, 127).to(torch.int8)
            return torch.cat([d.view(torch.uint8), q.view(torch.uint8)], -1).view(n, -1), (d, q)
        q = q.clamp_(-8, 7).to(torch.int8)
        u = (q + 8).view(torch.uint8)
        return torch.cat([d.view(torch.uint8), u[..., :16] | (u[..., 16:] << 4)], -1).view(n, -1), (d, q)
    s = b.view(n, k // 256, 8, 32)
    mn = (-s.amin(-1)).clamp_min_(0.0)
    sc = (s.amax(-1) + mn) / 15
    d, dm = ((v.amax(-1, keepdim=True) / 63).half() for v in (sc, mn))
    sc, mn = (_round(v / h.float().clamp_min(1e-30)).clamp_(0, 63) for v, h in ((sc, d), (mn, dm)))
    low = dm.float() * mn
    q = _round((s + low.unsqueeze(-1)) / (d.float() * sc).clamp_min(1e-30).unsqueeze(-1)).clamp_(0, 15).to(torch.uint8)
    a, m = sc.to(torch.uint8), mn.to(torch.uint8)
    scales = torch.cat([a[..., :4] | ((a[..., 4:] >> 4) << 6), m[..., :4] | ((m[..., 4:] >> 4) << 6),
                        (a[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)], -1)
    qs = (q[..., 0::2, :] | (q[..., 1::2, :] << 4)).reshape(n, k // 256, 128)
    return torch.cat([d.view(torch.uint8), dm.view(torch.uint8), scales, qs], -1).view(n, -1), (d, dm, a, m, q)


def _weight(dtype, n, k, seed, *path, std=0.02):
    return _encode(dtype, _normal((n, k), std, seed, *path))


def _qmm(dtype, n, k, seed, *path, std=0.02):
    blocks, _ = _weight(dtype, n, k, seed, *path, std=std)
    return QMatMul.from_qtensor(QTensor.from_blocks(blocks, (n, k), DTYPE[dtype], device=DEV))


def _weight64(dtype, n, k, seed, *path, std=0.02):
    """The decoded weight in 64 bits."""
    _, p = _weight(dtype, n, k, seed, *path, std=std)
    if dtype != "q4k":
        return (p[1].to(F64) * p[0].to(F64)).view(n, k)
    d, dm, a, m, q = (v.to(F64) for v in p)
    return ((d * a).unsqueeze(-1) * q - (dm * m).unsqueeze(-1)).view(n, k)


def _half_away(x):
    return torch.sign(x) * torch.floor(x.abs() + 0.5)


def _activation64(dtype, x):
    """The Q8 activation that the weight format's integer dot product multiplies with."""
    b = x.view(*x.shape[:-1], -1, BLOCK[dtype])
    if dtype == "q4k":
        top = torch.gather(b, -1, b.abs().argmax(-1, keepdim=True))
        inv = torch.where(top == 0, torch.zeros_like(top), -128.0 / top)
        q = _half_away(b * inv).clamp_max(127)
        return torch.where(inv == 0, torch.zeros_like(b), q / inv).view(x.shape)
    d = b.abs().amax(-1, keepdim=True) / 127
    q = torch.where(d == 0, torch.zeros_like(b), _half_away(b / d))
    return (q * d.to(torch.float16).to(F64)).view(x.shape)


def _x(case, seed):
    x = _normal((case["m"], case["k"]), 1.0, seed, 2)
    return x.bfloat16() if case["bf16"] else x


# ---- engines --------------------------------------------------------------------------

def _config(model, layers, max_seq, max_batch, whole=False):
    if model == "cv2":
        return cosyvoice2_lm_config(n_layers=layers, max_seq=max_seq, max_batch=max_batch)
    if whole:
        return fish_s2_slow_ar_config(n_layers=layers, max_seq=max_seq, max_batch=max_batch)
    # layers of the Fish block under the fast AR's 4096-row head, fed embeddings
    return fish_s2_slow_ar_config(n_layers=layers, max_seq=max_seq, max_batch=max_batch, n_codebooks=0, vocab=4096,
                                  tied_embedding=0, embed_rows=16)


def _dtype_name(cfg):
    return {int(v): k for k, v in DTYPE.items()}[cfg.weight_dtype]


def _widths(cfg):
    return cfg.n_heads * cfg.head_dim, cfg.n_kv_heads * cfg.head_dim


def _vector(cfg, layer, which, seed):
    ctx, kv = _widths(cfg)
    if which in (BQ, BK, BV, HEAD_BIAS):
        return _normal((cfg.vocab if which == HEAD_BIAS else ctx if which == BQ else kv,), 0.02, seed, layer, 50 + which)
    if which == EMBED:
        return _normal((cfg.vocab if cfg.tied_embedding else cfg.embed_rows, cfg.dim), 1.0, seed, 0, 50 + which)
    if which == CODEBOOK_EMBED:
        return _normal((cfg.n_codebooks * cfg.codebook_size, cfg.dim), 1.0, seed, 0, 50 + which)
    size = cfg.head_dim if which in (Q_NORM, K_NORM) else cfg.dim
    return 1.0 + _normal((size,), 0.1, seed, layer, 50 + which)


def _std(cfg, which):
    """The projections that write to the residual are scaled down by its number of terms, as
    is usual for initial weights."""
    return 0.02 / math.sqrt(2 * cfg.n_layers) if which in (WO, W2) else 0.02


def _projections(cfg):
    ctx, kv = _widths(cfg)
    return [(WQKV, ctx + 2 * kv, cfg.dim), (WO, cfg.dim, ctx), (W1, cfg.intermediate, cfg.dim),
            (W3, cfg.intermediate, cfg.dim), (W2, cfg.dim, cfg.intermediate)]


def _layer_vectors(cfg):
    return ([ATTN_NORM, FFN_NORM] + ([Q_NORM, K_NORM] if cfg.qk_norm else []) + ([BQ, BK, BV] if cfg.qkv_bias else []))


def _engine(cls, cfg, seed):
    lm, dt = cls(cfg, device=DEV), _dtype_name(cfg)
    for layer in range(cfg.n_layers):
        for which, n, k in _projections(cfg):
            lm.set_linear(layer, which, _qmm(dt, n, k, seed, layer, which, std=_std(cfg, which)))
        for which in _layer_vectors(cfg):
            lm.set_vector(layer, which, _vector(cfg, layer, which, seed))
    lm.set_linear(-1, HEAD, _qmm(dt, cfg.vocab, cfg.dim, seed, 999, HEAD))
    tables = [FINAL_NORM, EMBED] + ([HEAD_BIAS] if cfg.head_bias else []) + ([CODEBOOK_EMBED] if cfg.n_codebooks else [])
    for which in tables:
        lm.set_vector(-1, which, _vector(cfg, 0, which, seed))
    return lm


def _norm64(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.to(F64)


def _rope64(cfg, x, pos):
    half = cfg.head_dim // 2
    freq = 1.0 / torch.pow(torch.tensor(cfg.rope_theta, device=DEV), torch.arange(half, device=DEV) / half)
    ang = (pos.to(torch.float32)[:, None] * freq).to(F64)[:, None, :]  # the tables' f32 angles
    c, s = ang.cos(), ang.sin()
    if cfg.rope_interleaved:
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _decoder64(cfg, seed, streams, quantized):
    """Hidden rows (after the final norm) and head logits inputs of whole sequences in 64
    bits: streams is a list of [T, dim] inputs from position 0; quantized [sum T] marks the
    rows whose projections take Q8 activations."""
    dt, (ctx, kv), hd = _dtype_name(cfg), _widths(cfg), cfg.head_dim
    lens = [s.shape[0] for s in streams]
    h = torch.cat(streams).to(F64)
    pos = torch.cat([torch.arange(n, device=DEV) for n in lens])
    mask = quantized[:, None]

    def proj(x, layer, which, n, k):
        return torch.where(mask, _activation64(dt, x), x) @ _weight64(dt, n, k, seed, layer, which, std=_std(cfg, which)).t()

    for layer in range(cfg.n_layers):
        vec = {w: _vector(cfg, layer, w, seed) for w in _layer_vectors(cfg)}
        size = {w: (n, k) for w, n, k in _projections(cfg)}
        qkv = proj(_norm64(h, vec[ATTN_NORM], cfg.norm_eps), layer, WQKV, *size[WQKV])
        if cfg.qkv_bias:
            qkv = qkv + torch.cat([vec[BQ], vec[BK], vec[BV]]).to(F64)
        q, k, v = (t.reshape(h.shape[0], -1, hd) for t in qkv.split([ctx, kv, kv], -1))
        if cfg.qk_norm:
            q, k = _norm64(q, vec[Q_NORM], cfg.norm_eps), _norm64(k, vec[K_NORM], cfg.norm_eps)
        q, k = _rope64(cfg, q, pos), _rope64(cfg, k, pos)
        out, group, at = [], cfg.n_heads // cfg.n_kv_heads, 0
        for n in lens:
            qs, ks, vs = (t[at:at + n].transpose(0, 1) for t in (q, k, v))
            causal = torch.ones(n, n, dtype=torch.bool, device=DEV).triu(1)
            heads = []
            for i in range(cfg.n_heads):
                sc = (qs[i] @ ks[i // group].t()) / math.sqrt(hd)
                heads.append(torch.softmax(sc.masked_fill(causal, -math.inf), -1) @ vs[i // group])
            out.append(torch.cat(heads, -1))
            at += n
        h = h + proj(torch.cat(out), layer, WO, *size[WO])
        x = _norm64(h, vec[FFN_NORM], cfg.norm_eps)
        gate, up = proj(x, layer, W1, *size[W1]), proj(x, layer, W3, *size[W3])
        h = h + proj(torch.nn.functional.silu(gate) * up, layer, W2, *size[W2])
    return _norm64(h, _vector(cfg, 0, FINAL_NORM, seed), cfg.norm_eps)


def _head64(cfg, seed, rows, quantized):
    dt = _dtype_name(cfg)
    x = _activation64(dt, rows) if quantized else rows
    y = x @ _weight64(dt, cfg.vocab, cfg.dim, seed, 999, HEAD).t()
    return y + _vector(cfg, 0, HEAD_BIAS, seed).to(F64) if cfg.head_bias else y


def _prefill_quantized(cfg, rows):
    """Whether a prefill of that many rows multiplies Q8 activations (Q4_K takes its f16
    matrix product from 64 rows on)."""
    return cfg.weight_dtype != int(GgmlDType.Q4K) or rows < 64


# ---- families -------------------------------------------------------------------------

def _prompt_cfg(case):
    counts = _ints(case["counts"])
    return _config(case["model"], case["layers"], max(counts), len(counts))


def _prompt_embeds(case, cfg, seed):
    return [_normal((c, cfg.dim), 1.0, seed, 7, i) for i, c in enumerate(_ints(case["counts"]))]


def _decode_cfg(case):
    lens = _ints(case["lens"])
    return _config(case["model"], case["layers"], max(lens) + case["steps"] + 8, len(lens))


def _decode_inputs(case, cfg, seed):
    lens = _ints(case["lens"])
    prefix = [_normal((n, cfg.dim), 1.0, seed, 7, i) for i, n in enumerate(lens)]
    if case["model"] == "cv2":  # speech tokens
        ids = torch.randint(0, 6561, (case["steps"], len(lens), 1), generator=_gen(seed, 8), device=DEV, dtype=torch.int32)
        return prefix, ids
    return prefix, _normal((case["steps"], len(lens), cfg.dim), 1.0, seed, 8)


def _frame_cfg(case):
    lens = _ints(case["lens"])
    return _config("fish", 36, max(lens) + case["frames"] + 8, len(lens), whole=True)


def _fast_cfg(n):
    return fish_s2_fast_ar_config(max_batch=n)


def _frame_inputs(case, cfg, seed):
    """Prompt frames per stream and the frames fed to the timed steps: semantic id, then codes."""
    def frames(n, *path):
        g = _gen(seed, 9, *path)
        sem = torch.randint(cfg.semantic_begin, cfg.semantic_end + 1, (n, 1), generator=g, device=DEV)
        codes = torch.randint(0, cfg.codebook_size, (n, cfg.n_codebooks), generator=g, device=DEV)
        return torch.cat([sem, codes], 1).to(torch.int32)

    lens = _ints(case["lens"])
    return [frames(n, i) for i, n in enumerate(lens)], [frames(len(lens), 100 + f) for f in range(case["frames"])]


def prepare(case, seed):
    family = case["family"]
    if family == "linear":
        return {"case": case, "w": _qmm(case["dtype"], case["n"], case["k"], seed, 1), "x": _x(case, seed),
                "bias": _normal((case["n"],), 0.02, seed, 3) if case["bias"] else None}
    if family == "load":
        return {"case": case, "w": _normal((case["n"], case["k"]), 0.02, seed, 1)}
    if family == "prompt":
        cfg = _prompt_cfg(case)
        return {"case": case, "lm": _engine(Qwen2Lm if case["model"] == "cv2" else DecoderLM, cfg, seed),
                "embeds": _prompt_embeds(case, cfg, seed)}
    lens = _ints(case["lens"])
    if family == "decode":
        cfg = _decode_cfg(case)
        lm = _engine(Qwen2Lm if case["model"] == "cv2" else DecoderLM, cfg, seed)
        prefix, inputs = _decode_inputs(case, cfg, seed)
        DecoderLM.prefill(lm, embeds=prefix)
        state = {"case": case, "lm": lm, "lens": lens, "inputs": list(inputs)}
        if case["model"] == "cv2":
            state["sampler"] = RasSampler([seed + i for i in range(len(lens))], device=DEV)
            state["rng"] = state["sampler"].rng.clone()
        return state
    cfg = _frame_cfg(case)
    slow, fast = _engine(SlowAr, cfg, seed), _engine(FastAr, _fast_cfg(len(lens)), seed + 1)
    prefix, frames = _frame_inputs(case, cfg, seed)
    DecoderLM.prefill(slow, prompts=prefix)
    sampler = FishSampler([seed + i for i in range(len(lens))], SamplingParams(),
                          semantic=(cfg.semantic_begin, cfg.semantic_end, -1), device=DEV)
    n = len(lens)
    return {"case": case, "slow": slow, "fast": fast, "lens": lens, "frames": frames, "sampler": sampler,
            "rng": sampler.rng.clone(),
            # the loop's fixed buffers, as dualar.generate_frames keeps them
            "logits": torch.empty((n, cfg.vocab), device=DEV), "next": torch.empty(n, dtype=torch.int32, device=DEV),
            "hidden": torch.empty((n, cfg.dim), device=DEV),
            "drawn": torch.zeros((n, 1 + cfg.n_codebooks), dtype=torch.int32, device=DEV)}


def run(state):
    case = state["case"]
    family = case["family"]
    if family == "linear":
        return state["w"].forward(state["x"], state["bias"])
    if family == "load":
        return QTensor.quantize(state["w"], DTYPE[case["dtype"]]).data()
    if family == "prompt":
        lm = state["lm"]
        lm.reset(len(state["embeds"]))
        if case["all"] and len(state["embeds"]) == 1:
            return lm.forward_logits_cached(state["embeds"][0].unsqueeze(0))[0]
        logits, _, hidden = lm.prefill(embeds=state["embeds"], all_logits=case["all"])
        return [logits, hidden]
    if family == "decode":
        lm, out, ids = state["lm"], [], []
        lm.set_lengths(state["lens"])
        if case["model"] != "cv2":
            for x in state["inputs"]:
                logits, _, hidden = lm.step(embeds=x, graph=True, want_hidden=True)
                out += [logits, hidden]
            return out
        sampler = state["sampler"]
        sampler.rng.copy_(state["rng"])
        sampler.decoded_len.zero_()
        for x in state["inputs"]:
            logits, _ = lm.step(ids=x, graph=True)
            ids.append(sampler.sample(logits, ignore_eos=False))  # leaves log-probabilities in logits
            out.append(logits)
        return out + [torch.stack(ids)]
    slow, sampler, drawn, out, ids = state["slow"], state["sampler"], state["drawn"], [], []
    slow.set_lengths(state["lens"])
    sampler.rng.copy_(state["rng"])
    sampler.window_len.zero_()
    for frame in state["frames"]:
        logits, hidden = slow.slow_step_batch(frame, out=(state["logits"], state["next"], state["hidden"]))
        sampler.sample_semantic(logits, out=drawn, out_stride=drawn.stride(0))
        state["fast"].expand_batch(hidden, drawn[:, 0], sampler, codes=drawn[:, 1:])
        out += [logits.clone(), hidden.clone()]
        ids.append(drawn.clone())
    return out + [torch.stack(ids)]


def exact(case, seed):
    family = case["family"]
    if family == "linear":
        x = _x(case, seed).to(F64)
        if case["dtype"] != "q4k" or case["m"] < 64:
            x = _activation64(case["dtype"], x)
        y = x @ _weight64(case["dtype"], case["n"], case["k"], seed, 1).t()
        return y + _normal((case["n"],), 0.02, seed, 3).to(F64) if case["bias"] else y
    if family == "load":
        return None
    if family == "prompt":
        cfg, counts = _prompt_cfg(case), _ints(case["counts"])
        quantized = _prefill_quantized(cfg, sum(counts))
        rows = torch.full((sum(counts),), quantized, device=DEV)
        hidden = _decoder64(cfg, seed, _prompt_embeds(case, cfg, seed), rows)
        if case["all"]:
            logits = _head64(cfg, seed, hidden, quantized)
            return logits if len(counts) == 1 else [logits, hidden]
        last = torch.tensor(counts, device=DEV).cumsum(0) - 1
        return [_head64(cfg, seed, hidden[last], True), hidden[last]]
    lens = _ints(case["lens"])
    if family == "decode":
        cfg, steps = _decode_cfg(case), case["steps"]
        prefix, inputs = _decode_inputs(case, cfg, seed)
        if case["model"] == "cv2":
            inputs = _vector(cfg, 0, EMBED, seed)[inputs[..., 0].long()]
    else:
        cfg, steps = _frame_cfg(case), case["frames"]
        prompts, frames = _frame_inputs(case, cfg, seed)
        table, books = _vector(cfg, 0, EMBED, seed), _vector(cfg, 0, CODEBOOK_EMBED, seed)
        offset = torch.arange(cfg.n_codebooks, device=DEV) * cfg.codebook_size

        def embed(f):
            f = f.long()
            return (table[f[:, 0]].to(F64) + books[f[:, 1:] + offset].to(F64).sum(1)) / math.sqrt(cfg.n_codebooks + 1)

        prefix, inputs = [embed(p) for p in prompts], torch.stack([embed(f) for f in frames])
    streams = [torch.cat([p, inputs[:, i]]) for i, p in enumerate(prefix)]
    rows = torch.cat([torch.arange(n + steps, device=DEV) >= (0 if _prefill_quantized(cfg, sum(lens)) else n) for n in lens])
    hidden = _decoder64(cfg, seed, streams, rows)
    first = torch.cat([torch.zeros(1, dtype=torch.long, device=DEV),
                       torch.tensor([n + steps for n in lens], device=DEV).cumsum(0)[:-1]])
    out = []
    for t in range(steps):
        hid = hidden[first + torch.tensor(lens, device=DEV) + t]
        logits = _head64(cfg, seed, hid, True)
        if family == "frame":
            out += [logits, hid.unsqueeze(1)]
        elif case["model"] == "cv2":
            out.append(torch.log_softmax(logits, -1))
        else:
            out += [logits, hid]
    return out if family == "decode" and case["model"] != "cv2" else out + [None]


# ---- work -----------------------------------------------------------------------------

def _linear_work(dtype, n, k, m):
    return n * (k // BLOCK[dtype]) * BLOCK_BYTES[dtype], 2 * n * k * m


def _model_weights(cfg):
    """(layer bytes, layer multiply-adds x 2 per row, head bytes, head operations per row)."""
    dt, lb, lf = _dtype_name(cfg), 0, 0
    for _, n, k in _projections(cfg):
        b, f = _linear_work(dt, n, k, 1)
        lb, lf = lb + b * cfg.n_layers, lf + f * cfg.n_layers
    return (lb, lf) + _linear_work(dt, cfg.vocab, cfg.dim, 1)


def _steps_work(cfg, lens, steps):
    """Steps follow one another (each needs the one before), so each reads the weights and
    its streams' caches once."""
    (ctx, kv), n = _widths(cfg), len(lens)
    lb, lf, hb, hf = _model_weights(cfg)
    positions = sum(l + t + 1 for l in lens for t in range(steps))
    return {"bytes": steps * (lb + hb + 4 * n * (2 * cfg.dim + cfg.vocab)) + 8 * kv * cfg.n_layers * positions,
            "flops": steps * n * (lf + hf) + 4 * ctx * cfg.n_layers * positions}


def work(case):
    family = case["family"]
    if family == "linear":
        b, f = _linear_work(case["dtype"], case["n"], case["k"], case["m"])
        return {"bytes": b + case["m"] * (case["k"] * (2 if case["bf16"] else 4) + case["n"] * 4)
                + (case["n"] * 4 if case["bias"] else 0), "flops": f}
    if family == "load":  # Q4_K's search: five rounds of a least-squares step over every element
        b, _ = _linear_work(case["dtype"], case["n"], case["k"], 1)
        return {"bytes": case["n"] * case["k"] * 4 + b, "flops": case["n"] * case["k"] * (40 if case["dtype"] == "q4k" else 4)}
    if family == "prompt":
        cfg, counts = _prompt_cfg(case), _ints(case["counts"])
        (ctx, kv), T = _widths(cfg), sum(counts)
        lb, lf, hb, hf = _model_weights(cfg)
        rows = T if case["all"] else len(counts)
        pairs = sum(c * (c + 1) // 2 for c in counts)
        return {"bytes": lb + hb + 4 * (T * cfg.dim + rows * (cfg.vocab + cfg.dim)) + 8 * kv * T * cfg.n_layers,
                "flops": T * lf + rows * hf + 4 * ctx * pairs * cfg.n_layers}
    lens = _ints(case["lens"])
    if family == "decode":
        return _steps_work(_decode_cfg(case), lens, case["steps"])
    slow, fast = _steps_work(_frame_cfg(case), lens, case["frames"]), _steps_work(_fast_cfg(len(lens)), [0] * len(lens), 10)
    return {k: slow[k] + case["frames"] * fast[k] for k in slow}


def tolerance(case):
    """About four times what these show against `exact`, and where a model's outputs are
    compared, with its norm weights moved by half a unit in the last place (a one-ulp change
    of an activation moves some of the Q8 codes that the integer dot products take, and every
    layer behind it): the larger of the two."""
    family = case["family"]
    if family == "load":
        return "exact"
    if family == "linear":
        if case["dtype"] != "q4k":  # 1e-7 of f32 sums, 5e-5 where a Q8 code sits at a rounding tie
            return {"rel": 2e-4, "max": 7e-3}
        if case["m"] >= 64:  # 2.9e-4: f16 operands
            return {"rel": 1.2e-3, "max": 7e-3}
        return {"rel": 4.5e-4, "max": 7e-3}  # 1.1e-4: Q8_K codes at a rounding tie
    if family == "frame":
        # a moved logit changes a draw, and that draw the rest of its frame (0.4 to 0.8 of the ids seen)
        return {"rel": 9e-2, "max": 0.42, "differ": 0.95}
    if family == "decode":
        return {"rel": 1.6e-3, "max": 6e-3, "differ": 0.75} if case["model"] == "cv2" else {"rel": 7e-2, "max": 0.32}
    if case["model"] == "cv2":
        return {"rel": 2.2e-2, "max": 0.12}
    return {"rel": 7e-2, "max": 0.32} if sum(_ints(case["counts"])) < 64 else {"rel": 1.2e-2, "max": 5e-2}
