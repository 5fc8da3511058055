"""GPU parity of the on-device decode step (glue kernels + QMatMul GEMVs + driver)
against the CPU oracle of the reference's f32 decode step (oracle/model.py).

Two levels, both on identical quantized weights:

1. Op by op (teacher forcing).  The engine records every f32 intermediate of a step
   (sxq_lm_set_trace); each op is re-run by the oracle on the GPU's own input to that
   op.  Every projection inside the step (QKV, O, gate|up, down, head, with the
   activation quantization in front of it) must then match bit for bit, the
   embedding too, and each f32 glue op (RMSNorm, QK-RMSNorm + RoPE, attention over
   the GPU's cache, SiLU*mul) to GLUE_RTOL -- they differ only in summation order and
   expf's last bit.

2. End to end.  Over several layers the ~1e-7 glue differences occasionally move one
   activation across a Q8 rounding tie; in these random models one such flip moves
   the logits by up to ~2e-2 (measured on the oracle alone).  So every step must agree
   to LOGIT_RTOL_FLIP, and most steps -- all, barring a flip -- to LOGIT_RTOL.
"""
import os

import numpy as np
import pytest
import torch

from syrinx_amd import GgmlDType, QMatMul, QTensor
from syrinx_amd import decoder as D

pytestmark = pytest.mark.gpu

GLUE_RTOL = 4e-6        # |gpu - oracle| <= GLUE_RTOL * (|oracle| + max |oracle|) for f32 glue ops
LOGIT_RTOL = 1e-5       # max |gpu - oracle| / max |oracle| of a step's logits, no Q8 flip
LOGIT_RTOL_FLIP = 5e-2  # the same bound for any step (one activation one Q8 step apart)
TIGHT_FRACTION = 0.6    # share of a test's steps that must meet LOGIT_RTOL (one flip always allowed)
KV_ATOL = 2e-5          # post-RoPE key rows (unit-RMS values), absolute

class _Tally:
    """Steps of one test in the tight (no Q8 flip) and flip regimes; each test checks its
    own tally, so the check does not depend on which tests ran before."""

    def __init__(self):
        self.tight = 0
        self.flip = 0

    def mostly_tight(self):
        n = self.tight + self.flip
        assert n > 0 and self.flip <= max(1, int((1.0 - TIGHT_FRACTION) * n)), (self.tight, self.flip)


def _check(got, orc, want, what, tally=None):
    err = _rel(got, want)
    tight = err <= LOGIT_RTOL
    if tally is not None:
        if tight:
            tally.tight += 1
        else:
            tally.flip += 1
    print(f"{what}: rel err {err:.2e} (smallest quantization margin {orc.margin:.1e})")
    assert err <= LOGIT_RTOL_FLIP, (what, err, orc.margin)


@pytest.fixture(scope="module")
def cuda():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm GPU")
    return torch.device("cuda:0")


@pytest.fixture(scope="module")
def model_oracle():
    import model  # oracle/model.py, the CPU oracle of a decode step
    return model


def _build(cfg, cuda, seed, n_streams, cls=D.DecoderLM, dense_table=True):
    """Random weights -> GPU engine (of class cls) and the same blocks/vectors for the oracle.
    A tied model also gets its dense input table (the f32 rows its head was quantized
    from) unless dense_table is False (then it embeds through the dequantized head rows)."""
    rng = np.random.default_rng(seed)
    dt = GgmlDType(cfg.weight_dtype)
    lm = cls(cfg, device=cuda)
    W = {}
    hd, nh, nkv = cfg.head_dim, cfg.n_heads, cfg.n_kv_heads
    qkv_n = (nh + 2 * nkv) * hd

    def lin(n, k, key, slot, layer):
        w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
        qt = QTensor.quantize(torch.from_numpy(w).to(cuda), dt)
        blocks = qt.data().cpu().numpy().reshape(n, -1)
        lm.set_linear(layer, slot, QMatMul.from_qtensor(qt))
        W[key] = blocks
        return w

    def vec(n, key, slot, layer, mean, std):
        v = (mean + rng.standard_normal(n) * std).astype(np.float32)
        lm.set_vector(layer, slot, torch.from_numpy(v))
        W[key] = v

    for l in range(cfg.n_layers):
        if cfg.qkv_bias:  # Qwen2: three projections fused on upload
            lin(nh * hd, cfg.dim, ("wq", l), D.WQ, l)
            lin(nkv * hd, cfg.dim, ("wk", l), D.WK, l)
            lin(nkv * hd, cfg.dim, ("wv", l), D.WV, l)
            W[("wqkv", l)] = np.concatenate([W.pop(("wq", l)), W.pop(("wk", l)), W.pop(("wv", l))])
            vec(nh * hd, ("bq", l), D.BQ, l, 0.0, 0.02)
            vec(nkv * hd, ("bk", l), D.BK, l, 0.0, 0.02)
            vec(nkv * hd, ("bv", l), D.BV, l, 0.0, 0.02)
            W[("bqkv", l)] = np.concatenate([W.pop(("bq", l)), W.pop(("bk", l)), W.pop(("bv", l))])
        else:
            lin(qkv_n, cfg.dim, ("wqkv", l), D.WQKV, l)
        lin(cfg.dim, nh * hd, ("wo", l), D.WO, l)
        lin(cfg.intermediate, cfg.dim, ("w1", l), D.W1, l)
        lin(cfg.intermediate, cfg.dim, ("w3", l), D.W3, l)
        lin(cfg.dim, cfg.intermediate, ("w2", l), D.W2, l)
        vec(cfg.dim, ("attn_norm", l), D.ATTN_NORM, l, 1.0, 0.1)
        vec(cfg.dim, ("ffn_norm", l), D.FFN_NORM, l, 1.0, 0.1)
        if cfg.qk_norm:
            vec(hd, ("q_norm", l), D.Q_NORM, l, 1.0, 0.1)
            vec(hd, ("k_norm", l), D.K_NORM, l, 1.0, 0.1)
    head_w = lin(cfg.vocab, cfg.dim, "head", D.HEAD, -1)
    vec(cfg.dim, "final_norm", D.FINAL_NORM, -1, 1.0, 0.1)
    if cfg.head_bias:
        vec(cfg.vocab, "head_bias", D.HEAD_BIAS, -1, 0.0, 0.02)
    if not cfg.tied_embedding:
        rows = cfg.embed_rows or cfg.vocab
        vec(rows * cfg.dim, "embed", D.EMBED, -1, 0.0, 0.5)
        W["embed"] = W["embed"].reshape(rows, cfg.dim)
    elif dense_table:  # the tied head's source rows: the embedding gathers them (slow_ar.rs:117)
        lm.set_vector(-1, D.EMBED, torch.from_numpy(head_w.reshape(-1)))
        W["embed"] = head_w
    if cfg.n_codebooks:
        vec(cfg.n_codebooks * cfg.codebook_size * cfg.dim, "codebook", D.CODEBOOK_EMBED, -1, 0.0, 0.5)
        W["codebook"] = W["codebook"].reshape(-1, cfg.dim)
    if getattr(cfg, "o_bias", 0):
        for l in range(cfg.n_layers):
            vec(cfg.dim, ("bo", l), D.BO, l, 0.0, 0.02)
    return lm, W


def _build_dev(cfg, cuda, seed):
    """Like _build, with the projection weights drawn on the GPU (full-size models):
    N(0, 0.02) from a seeded torch generator, quantized by QTensor.quantize, the same
    canonical blocks handed to the engine and to the oracle."""
    dt = GgmlDType(cfg.weight_dtype)
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=cuda).manual_seed(seed)
    lm = D.DecoderLM(cfg, device=cuda)
    W = {}
    hd, nh, nkv = cfg.head_dim, cfg.n_heads, cfg.n_kv_heads
    qkv_n = (nh + 2 * nkv) * hd

    def lin(n, k, key, slot, layer, keep=False):
        w = torch.randn(n, k, device=cuda, generator=gen) * 0.02
        qt = QTensor.quantize(w, dt)
        lm.set_linear(layer, slot, QMatMul.from_qtensor(qt))
        W[key] = qt.data().cpu().numpy().reshape(n, -1)
        return w if keep else None

    def vec(n, key, slot, layer, mean, std):
        v = (mean + rng.standard_normal(n) * std).astype(np.float32)
        lm.set_vector(layer, slot, torch.from_numpy(v))
        W[key] = v

    for l in range(cfg.n_layers):
        if cfg.qkv_bias:
            lin(nh * hd, cfg.dim, ("wq", l), D.WQ, l)
            lin(nkv * hd, cfg.dim, ("wk", l), D.WK, l)
            lin(nkv * hd, cfg.dim, ("wv", l), D.WV, l)
            W[("wqkv", l)] = np.concatenate([W.pop(("wq", l)), W.pop(("wk", l)), W.pop(("wv", l))])
            b = [(rng.standard_normal(r) * 0.02).astype(np.float32) for r in (nh * hd, nkv * hd, nkv * hd)]
            for slot, v in zip((D.BQ, D.BK, D.BV), b):
                lm.set_vector(l, slot, torch.from_numpy(v))
            W[("bqkv", l)] = np.concatenate(b)
        else:
            lin(qkv_n, cfg.dim, ("wqkv", l), D.WQKV, l)
        lin(cfg.dim, nh * hd, ("wo", l), D.WO, l)
        lin(cfg.intermediate, cfg.dim, ("w1", l), D.W1, l)
        lin(cfg.intermediate, cfg.dim, ("w3", l), D.W3, l)
        lin(cfg.dim, cfg.intermediate, ("w2", l), D.W2, l)
        vec(cfg.dim, ("attn_norm", l), D.ATTN_NORM, l, 1.0, 0.1)
        vec(cfg.dim, ("ffn_norm", l), D.FFN_NORM, l, 1.0, 0.1)
        if cfg.qk_norm:
            vec(hd, ("q_norm", l), D.Q_NORM, l, 1.0, 0.1)
            vec(hd, ("k_norm", l), D.K_NORM, l, 1.0, 0.1)
    head_w = lin(cfg.vocab, cfg.dim, "head", D.HEAD, -1, keep=bool(cfg.tied_embedding))
    vec(cfg.dim, "final_norm", D.FINAL_NORM, -1, 1.0, 0.1)
    if cfg.head_bias:
        vec(cfg.vocab, "head_bias", D.HEAD_BIAS, -1, 0.0, 0.02)
    if not cfg.tied_embedding:
        rows = cfg.embed_rows or cfg.vocab
        vec(rows * cfg.dim, "embed", D.EMBED, -1, 0.0, 0.5)
        W["embed"] = W["embed"].reshape(rows, cfg.dim)
    else:  # the dense table stays on the device; the oracle reads the rows it gathers
        lm.set_vector(-1, D.EMBED, head_w.reshape(-1))
        W["embed"] = _DeviceRows(head_w)
    if cfg.n_codebooks:
        vec(cfg.n_codebooks * cfg.codebook_size * cfg.dim, "codebook", D.CODEBOOK_EMBED, -1, 0.0, 0.5)
        W["codebook"] = W["codebook"].reshape(-1, cfg.dim)
    return lm, W


class _DeviceRows:
    """Rows of a device table, copied to the host one at a time (a 1.6 GB table stays put)."""

    def __init__(self, t):
        self.t = t

    def __getitem__(self, i):
        return self.t[int(i)].float().cpu().numpy()


def _prefill(lm, orc, cfg, lengths, seed):
    lm.kv_fill_random(lengths, seed=seed)
    for s, L in enumerate(lengths):
        for l in range(cfg.n_layers):
            for g in range(cfg.n_kv_heads):
                if L:
                    k, v = lm.read_kv(l, s, g, 0, L)
                    orc.load_prefix(s, l, g, k.cpu().numpy(), v.cpu().numpy())


def _rel(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-30))


def _fish_small(n_layers=2, max_batch=1, dtype=GgmlDType.Q4K, **kw):
    return D.fish_s2_slow_ar_config(n_layers=n_layers, max_seq=96, max_batch=max_batch, dtype=dtype, vocab=4096,
                                    n_codebooks=10, codebook_size=64, semantic_begin=3000, semantic_end=4095, **kw)


def _frames(rng, n, cfg):
    f = np.zeros((n, 1 + cfg.n_codebooks), np.int32)
    f[:, 0] = rng.integers(0, cfg.vocab, n)
    f[: max(1, n // 2), 0] = rng.integers(cfg.semantic_begin, cfg.semantic_end + 1, max(1, n // 2))
    if cfg.n_codebooks:
        f[:, 1:] = rng.integers(0, cfg.codebook_size, (n, cfg.n_codebooks))
    return f



def _bits_equal(got, want, what):
    got = np.asarray(got, np.float32)
    want = np.asarray(want, np.float32)
    same = (got.view(np.uint32) == want.view(np.uint32)) | ((got == 0) & (want == 0))
    assert same.all(), f"{what}: {(~same).sum()} of {same.size} differ, max |d| {np.abs(got - want).max():.3e}"


def _glue_close(got, want, what):
    got = np.asarray(got, np.float64)
    want = np.asarray(want, np.float64)
    tol = GLUE_RTOL * (np.abs(want) + np.abs(want).max())
    bad = np.abs(got - want) > tol
    assert not bad.any(), f"{what}: {bad.sum()} of {bad.size} beyond {GLUE_RTOL:g}, max rel {np.abs(got - want).max() / np.abs(want).max():.2e}"


_ABS_W = {}


def _split_close(ora, got, base, o, x, W, key, dt, what):
    """got = base + o' where o' is the projection o computed with its K split over
    workgroups (the same products, the class chains added in another association): within
    1e-6 * sum_k |w_k x_k| of o per output, plus the residual add's own rounding.  Prints
    the largest error seen, relative to sum |w x|."""
    k = x.shape[-1]
    cache = (id(W), key)
    if cache not in _ABS_W:
        _ABS_W[cache] = np.abs(ora.dequantize(dt, W[key], k).reshape(-1, k)).astype(np.float64)
    s = _ABS_W[cache] @ np.abs(np.asarray(x, np.float64))
    want = (base + o).astype(np.float32)
    d = np.abs(np.asarray(got, np.float64) - want)
    print(f"{what}: split-K max |d| / sum|w x| = {np.max(d / s):.2e}")
    assert (d <= 1e-6 * s + 2.0 ** -23 * np.abs(want)).all(), (what, float(np.max(d / s)))


def _replay_step(ora, lm, cfg, W, tr, s, pos, frame=None, split=False):
    """Check every op of one traced step of stream s (placed at position pos); with split,
    the O and down projections (the 16-row matrix-core GEMV with K split over workgroups)
    are held to _split_close instead of bit equality."""
    dt = int(cfg.weight_dtype)
    hd, nh, nkv = cfg.head_dim, cfg.n_heads, cfg.n_kv_heads
    G = nh // nkv
    if frame is not None:
        import model
        orc = model.OracleDecoder(cfg, W, 1)
        _bits_equal(tr["embed"][s], orc.embed(frame), "embedding")
    h_in = tr["embed"][s]
    cos, sin = (ora.rope_tables_interleaved(pos + 1, hd, cfg.rope_theta) if cfg.rope_interleaved
                else ora.rope_tables_half(pos + 1, hd, cfg.rope_theta))
    rope = ora.rope_interleaved if cfg.rope_interleaved else ora.rope_half
    for l, T in enumerate(tr["layers"]):
        T = {k: v[s] for k, v in T.items()}
        tag = f"stream {s} layer {l}"
        _glue_close(T["hn_attn"], ora.rms_norm(h_in, W[("attn_norm", l)], cfg.norm_eps), f"{tag} attention RMSNorm")
        qkv = ora.matmul(dt, T["hn_attn"][None], W[("wqkv", l)])[0]
        if cfg.qkv_bias:
            qkv = (qkv + W[("bqkv", l)]).astype(np.float32)
        _bits_equal(T["qkv"], qkv, f"{tag} qkv projection")
        q = T["qkv"][: nh * hd].reshape(nh, hd)
        k = T["qkv"][nh * hd:(nh + nkv) * hd].reshape(nkv, hd)
        v = T["qkv"][(nh + nkv) * hd:].reshape(nkv, hd)
        if cfg.qk_norm:
            q = np.stack([ora.rms_norm(q[i], W[("q_norm", l)], cfg.norm_eps) for i in range(nh)])
            k = np.stack([ora.rms_norm(k[i], W[("k_norm", l)], cfg.norm_eps) for i in range(nkv)])
        _glue_close(T["q"], rope(q, cos[pos], sin[pos]).reshape(-1), f"{tag} QK-norm + RoPE (q)")
        kr = rope(k, cos[pos], sin[pos])
        ctx = np.zeros(nh * hd, np.float32)
        for g in range(nkv):
            kc, vc = lm.read_kv(l, s, g, 0, pos + 1)
            kc, vc = kc.cpu().numpy(), vc.cpu().numpy()
            _glue_close(kc[pos], kr[g], f"{tag} QK-norm + RoPE (k, head {g})")
            _bits_equal(vc[pos], v[g], f"{tag} value append (head {g})")
            for i in range(g * G, (g + 1) * G):
                ctx[i * hd:(i + 1) * hd] = ora.attend_one(T["q"][i * hd:(i + 1) * hd], kc, vc)
        _glue_close(T["ctx"], ctx, f"{tag} attention")
        o = ora.matmul(dt, T["ctx"][None], W[("wo", l)])[0]
        if getattr(cfg, "o_bias", 0):
            o = (o + W[("bo", l)]).astype(np.float32)
        if split:
            _split_close(ora, T["h_mid"], h_in, o, T["ctx"], W, ("wo", l), dt, f"{tag} O projection + residual")
        else:
            _bits_equal(T["h_mid"], (h_in + o).astype(np.float32), f"{tag} O projection + residual")
        _glue_close(T["hn_ffn"], ora.rms_norm(T["h_mid"], W[("ffn_norm", l)], cfg.norm_eps), f"{tag} FFN RMSNorm")
        gu = np.concatenate([ora.matmul(dt, T["hn_ffn"][None], W[("w1", l)])[0],
                             ora.matmul(dt, T["hn_ffn"][None], W[("w3", l)])[0]])
        _bits_equal(T["gu"], gu, f"{tag} gate|up projection")
        I = cfg.intermediate
        _glue_close(T["act"], ora.silu_mul(T["gu"][:I], T["gu"][I:]), f"{tag} SiLU*mul")
        o2 = ora.matmul(dt, T["act"][None], W[("w2", l)])[0]
        if split:
            _split_close(ora, T["h_out"], T["h_mid"], o2, T["act"], W, ("w2", l), dt, f"{tag} down projection + residual")
        else:
            _bits_equal(T["h_out"], (T["h_mid"] + o2).astype(np.float32), f"{tag} down projection + residual")
        h_in = T["h_out"]
    _glue_close(tr["final_hn"][s], ora.rms_norm(h_in, W["final_norm"], cfg.norm_eps), f"stream {s} final RMSNorm")
    logits = ora.matmul(dt, tr["final_hn"][s][None], W["head"])[0]
    if cfg.head_bias:
        logits = (logits + W["head_bias"]).astype(np.float32)
    return logits


# kinds ending in "_3k" force the three-kernel attention (RoPE/append, split partials,
# merge) instead of the fused kernel; "long" has 51 attention splits, more than the
# fused kernel stages in one chunk of its merge.
# "fish_bias": a checkpoint with wqkv.bias and wo.bias (both detected from the tensors,
# crates/syrinx-fish/src/s2/slow_ar.rs:91-93); "fish_untied": an output.weight head with
# the MCF embedding over the separate dense table; "fish_headrows": a tied model given no
# dense table (the embedding dequantizes the head rows).
@pytest.mark.parametrize("kind", ["fish_q4k", "fish_q8_0", "cv2_q8_0", "cv2_q4_0", "ragged", "fish_q4k_3k",
                                  "ragged_3k", "cv2_q8_0_3k", "long", "fish_bias", "fish_untied", "fish_headrows"])
def test_every_op_of_a_step_matches_oracle(cuda, ora, kind, monkeypatch):
    if kind.endswith("_3k"):
        monkeypatch.setenv("SXQ_ATTN_UNFUSED", "1")  # read when the engine is created
    if kind == "fish_bias":
        cfg = _fish_small(qkv_bias=1, o_bias=1)
        lengths = [40]
    elif kind == "fish_untied":
        cfg = _fish_small(tied_embedding=0)
        lengths = [40]
    elif kind.startswith("fish"):
        cfg = _fish_small(dtype=GgmlDType.Q8_0 if kind == "fish_q8_0" else GgmlDType.Q4K)
        lengths = [40]
    elif kind.startswith("cv2"):
        cfg = D.cosyvoice2_lm_config(n_layers=2, max_seq=96, dtype=GgmlDType.Q4_0 if kind == "cv2_q4_0" else GgmlDType.Q8_0)
        lengths = [70]  # two attention splits
    elif kind == "long":
        cfg = D.fish_s2_slow_ar_config(n_layers=1, max_seq=1664, vocab=4096, n_codebooks=10, codebook_size=64,
                                       semantic_begin=3000, semantic_end=4095)
        lengths = [1600]
    else:
        cfg = _fish_small(n_layers=1, max_batch=4)
        lengths = [5, 70, 17, 0]
    n = len(lengths)
    lm, W = _build(cfg, cuda, 21, n, dense_table=kind != "fish_headrows")
    lm.kv_fill_random(lengths, seed=22)
    lm.enable_trace()
    rng = np.random.default_rng(23)
    for step in range(2):
        if kind.startswith("cv2") and step == 0:
            emb = rng.standard_normal((n, cfg.dim)).astype(np.float32)
            logits, _ = lm.step(embeds=torch.from_numpy(emb))
            frames = [None] * n
        else:
            fr = _frames(rng, n, cfg) if not kind.startswith("cv2") else rng.integers(0, cfg.vocab, (n, 1)).astype(np.int32)
            logits, _ = lm.step(ids=torch.from_numpy(fr))
            frames = list(fr)
        tr = lm.trace(n)
        got = logits.cpu().numpy()
        for s in range(n):
            want = _replay_step(ora, lm, cfg, W, tr, s, lengths[s] + step, frame=frames[s])
            _bits_equal(got[s], want, f"{kind} stream {s} head projection")


def test_fish_slow_ar_step_matches_oracle(cuda, model_oracle):
    tally = _Tally()
    cfg = _fish_small()
    lm, W = _build(cfg, cuda, 1, 1)
    orc = model_oracle.OracleDecoder(cfg, W, 1)
    _prefill(lm, orc, cfg, [40], seed=3)
    rng = np.random.default_rng(2)
    for step in range(4):
        fr = _frames(rng, 1, cfg)
        logits, nxt = lm.step(ids=torch.from_numpy(fr))
        got = logits.cpu().numpy()[0]
        want = orc.step_one(0, frame=fr[0])
        _check(got, orc, want, f"fish step {step}", tally)
        assert int(nxt[0]) == int(np.argmax(got))
        # the rows this step appended (post QK-RMSNorm + RoPE keys, raw values); after a
        # Q8 flip they carry its effect, so they are compared on flip-free steps only.
        # Then the oracle takes the engine's rows, so a flip in one step does not carry
        # into the caches of the next (each step is judged on its own).
        pos = 40 + step
        tight = _rel(got, want) <= LOGIT_RTOL
        for l in range(cfg.n_layers):
            for g in range(cfg.n_kv_heads):
                k, v = lm.read_kv(l, 0, g, pos, 1)
                k, v = k.cpu().numpy()[0], v.cpu().numpy()[0]
                if tight:
                    np.testing.assert_allclose(k, orc.k[0][l][g][pos], rtol=0, atol=KV_ATOL)
                    np.testing.assert_allclose(v, orc.v[0][l][g][pos], rtol=0, atol=KV_ATOL)
                orc.k[0][l][g][pos] = k
                orc.v[0][l][g][pos] = v
    assert lm.lengths(1) == [44]
    tally.mostly_tight()


@pytest.mark.parametrize("dtype", [GgmlDType.Q8_0, GgmlDType.Q4_0])
def test_cosyvoice2_lm_step_matches_oracle(cuda, model_oracle, dtype):
    tally = _Tally()
    cfg = D.cosyvoice2_lm_config(n_layers=2, max_seq=64, dtype=dtype)
    lm, W = _build(cfg, cuda, 4, 1)
    orc = model_oracle.OracleDecoder(cfg, W, 1)
    _prefill(lm, orc, cfg, [17], seed=5)
    rng = np.random.default_rng(6)
    for step in range(2):
        emb = rng.standard_normal((1, cfg.dim)).astype(np.float32)
        logits, _ = lm.step(embeds=torch.from_numpy(emb))
        got = logits.cpu().numpy()[0]
        want = orc.step_one(0, embed=emb[0])
        _check(got, orc, want, f"cv2 {dtype.name} step {step}", tally)
    # token-id path through the dense speech-embedding table
    tok = np.array([[1234]], np.int32)
    logits, _ = lm.step(ids=torch.from_numpy(tok))
    _check(logits.cpu().numpy()[0], orc, orc.step_one(0, frame=tok[0]), f"cv2 {dtype.name} token step", tally)
    tally.mostly_tight()


# 4 streams: the task-split GEMV; 7 streams: Q4_K projections on the matrix-core GEMV
@pytest.mark.parametrize("lengths", [[5, 70, 17, 0], [5, 70, 17, 0, 33, 1, 48]])
def test_ragged_batch_matches_per_stream_oracle(cuda, model_oracle, lengths):
    tally = _Tally()
    B = len(lengths)
    cfg = _fish_small(n_layers=1, max_batch=B)
    lm, W = _build(cfg, cuda, 7, B)
    orc = model_oracle.OracleDecoder(cfg, W, B)
    _prefill(lm, orc, cfg, lengths, seed=8)
    rng = np.random.default_rng(9)
    for step in range(2):
        fr = _frames(rng, B, cfg)
        logits, _ = lm.step(ids=torch.from_numpy(fr))
        got = logits.cpu().numpy()
        for s in range(B):
            want = orc.step_one(s, frame=fr[s])
            _check(got[s], orc, want, f"ragged step {step} stream {s} (len {lengths[s] + step})", tally)
    assert lm.lengths(B) == [L + 2 for L in lengths]
    tally.mostly_tight()


# (250, 3): the longer stream crosses 256 positions, where the step's attention grid grows
# by a bucket of four 64-position splits (a graph per bucket).
@pytest.mark.parametrize("lens,steps", [((12, 30), 4), ((250, 3), 10)])
def test_graph_replay_equals_eager_and_feeds_back_argmax(cuda, lens, steps):
    cfg = _fish_small(n_layers=2, max_batch=2)
    cfg.max_seq = 320
    res = {}
    for mode in ("eager", "graph"):
        lm, _ = _build(cfg, cuda, 10, 2)
        lm.kv_fill_random(list(lens), seed=11)
        fr = _frames(np.random.default_rng(12), 2, cfg)
        outs = []
        logits, nxt = lm.step(ids=torch.from_numpy(fr), graph=(mode == "graph"))
        outs.append(logits.cpu().numpy())
        for _ in range(steps):  # greedy: reuse the device-side argmax
            _ = torch.zeros(1000, device=cuda).sum().item()  # eager work between replays
            logits2, nxt2 = lm.step(n=2, graph=(mode == "graph"))
            torch.cuda.synchronize()
            outs.append(logits2.cpu().numpy())
            assert (nxt2.cpu().numpy() == np.argmax(outs[-1], axis=1)).all()
        res[mode] = outs
        assert lm.lengths(2) == [L + steps + 1 for L in lens]
    for a, b in zip(res["eager"], res["graph"]):
        np.testing.assert_array_equal(a, b)


PAIR_KINDS = {  # the SwiGLU pair at each weight type: Qwen3-4B width (w1|w3 19456 x 2560, w2 2560 x 9728)
    "fish_q4k": ("fish", GgmlDType.Q4K),       # and the CosyVoice2 width (9728 x 896, 896 x 4864)
    "fish_q8_0": ("fish", GgmlDType.Q8_0),     # 12 task rounds per gate|up tile
    "fish_q4_0": ("fish", GgmlDType.Q4_0),
    "cv2_q8_0": ("cv2", GgmlDType.Q8_0),
    "cv2_q4_0": ("cv2", GgmlDType.Q4_0),       # the dtype the reference's load_quantized ships
}


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("kind", sorted(PAIR_KINDS))
def test_swiglu_pair_equals_three_launches(cuda, monkeypatch, graph, kind):
    """One decode row: the gate|up GEMV with the SwiGLU epilogue and the down GEMV that
    quantizes in its prologue give the bits of GEMV + SiLU*mul kernel + GEMV, for Q4_K,
    Q8_0 and Q4_0 weights.  The pair's own output row (read_state 5) shows which path ran:
    silu(g) * u of the step's gate|up row with the pair, untouched zeros without."""
    if os.environ.get("SXQ_GEMV_WG"):
        pytest.skip("SXQ_GEMV_WG regrids the GEMVs (read once per process): the pair's tiles are laid out "
                    "for the default grid, so the engine runs three launches")
    cfg = _small_cfg(kind, 2)
    res = {}
    for mode in ("pair", "three"):
        if mode == "three":
            monkeypatch.setenv("SXQ_SWIGLU_UNFUSED", "1")  # read when the engine is created
        else:
            monkeypatch.delenv("SXQ_SWIGLU_UNFUSED", raising=False)
        lm = D.DecoderLM(cfg, device=cuda)
        assert bool(lm.paths() & lm.PATH_SWIGLU) == (mode == "pair"), lm.paths()
        lm.init_random(seed=41, std=0.02)
        lm.kv_fill_random([33], seed=42)
        fr = _first_ids(kind, cfg, np.random.default_rng(43))
        logits, _ = lm.step(ids=torch.from_numpy(fr), graph=graph)
        outs = [logits.cpu().numpy()]
        for _ in range(3):
            logits, _ = lm.step(n=1, graph=graph)
            outs.append(logits.cpu().numpy())
        res[mode] = outs
        act = lm.read_state(5).cpu().numpy()[0]
        if mode == "pair":
            gu = lm.read_state(3).cpu().numpy()[0].astype(np.float64)
            g, u = gu[: cfg.intermediate], gu[cfg.intermediate:]
            np.testing.assert_allclose(act, g / (1.0 + np.exp(-g)) * u, rtol=1e-5, atol=1e-7)
            assert np.abs(act).max() > 0
        else:
            assert not act.any(), "the unfused engine ran the pair"
    for a, b in zip(res["pair"], res["three"]):
        np.testing.assert_array_equal(a, b)


def _small_cfg(kind, n_layers):
    model, dt = PAIR_KINDS[kind]
    if model == "fish":
        return _fish_small(n_layers=n_layers, dtype=dt)
    return D.cosyvoice2_lm_config(n_layers=n_layers, max_seq=96, dtype=dt)


def _first_ids(kind, cfg, rng):
    if PAIR_KINDS[kind][0] == "fish":
        return _frames(rng, 1, cfg)
    return rng.integers(0, cfg.vocab, (1, 1)).astype(np.int32)


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("kv", [33, 200])
@pytest.mark.parametrize("kind", sorted(PAIR_KINDS))
def test_attention_and_o_projection_in_one_launch_equals_two(cuda, monkeypatch, graph, kv, kind):
    """One decode row: attention with the O projection's workgroups in the same launch
    (waiting on per-layer ready counters, which consecutive layers zero for each other)
    gives the bits of the attention launch followed by the O-projection GEMV -- with one
    attention split (kv 33) and with a merge of four (kv 200), over three layers and five
    steps, so every counter is used, zeroed and reused; Q4_K (Q8_K context slices) and
    Q8_0 / Q4_0 (Q8_0 slices) projections, at the Qwen3-4B and the CosyVoice2 shapes."""
    cfg = _small_cfg(kind, 3)
    cfg.max_seq = 256
    res = {}
    for mode in ("one", "two"):
        if mode == "two":
            monkeypatch.setenv("SXQ_ATTN_WO_UNFUSED", "1")  # read when the engine is created
        else:  # the fused launch needs the fused attention as well
            monkeypatch.delenv("SXQ_ATTN_WO_UNFUSED", raising=False)
            monkeypatch.delenv("SXQ_ATTN_UNFUSED", raising=False)
        lm = D.DecoderLM(cfg, device=cuda)
        assert bool(lm.paths() & lm.PATH_ATTN_WO) == (mode == "one"), lm.paths()
        lm.init_random(seed=51, std=0.02)
        lm.kv_fill_random([kv], seed=52)
        fr = _first_ids(kind, cfg, np.random.default_rng(53))
        logits, _ = lm.step(ids=torch.from_numpy(fr), graph=graph)
        outs = [logits.cpu().numpy()]
        for _ in range(4):
            _ = torch.zeros(1000, device=cuda).sum().item()  # eager work between replays
            logits, _ = lm.step(n=1, graph=graph)
            outs.append(logits.cpu().numpy())
        assert lm.lengths(1) == [kv + 5]
        res[mode] = outs
    for a, b in zip(res["one"], res["two"]):
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("kind,cut", [("fish_q4k", 40), ("cv2_q8_0", 40), ("cv2_q8_0", 100)])
def test_graph_replayed_at_shorter_lengths_than_captured(cuda, kind, cut):
    """A step captured at a long length and replayed after the lengths were cut (the
    attention grid and every length-dependent choice were fixed at capture; the splits
    past the new length now idle) gives the bits of an eager step at the new lengths --
    down to one split (cut 40, no merge) and to two (cut 100), at the Qwen3-4B and the
    CosyVoice2 shapes."""
    cfg = _small_cfg(kind, 2)
    cfg.max_seq = 256
    fr = _first_ids(kind, cfg, np.random.default_rng(73))
    outs = []
    for graph in (True, False):
        lm = D.DecoderLM(cfg, device=cuda)
        lm.init_random(seed=71, std=0.02)
        lm.kv_fill_random([200], seed=72)
        if graph:
            lm.step(ids=torch.from_numpy(fr), graph=True)  # captured with four splits per head group
        lm.set_lengths([cut])
        logits, _ = lm.step(ids=torch.from_numpy(fr), graph=graph)
        outs.append(logits.cpu().numpy())
        assert lm.lengths(1) == [cut + 1]
    assert np.isfinite(outs[0]).all()
    np.testing.assert_array_equal(outs[0], outs[1])


def test_full_cache_is_an_error(cuda):
    cfg = _fish_small(n_layers=1)
    cfg.max_seq = 8
    lm = D.DecoderLM(cfg, device=cuda)
    lm.init_random(seed=1)
    lm.set_lengths([7])
    lm.step(ids=torch.zeros((1, 11), dtype=torch.int32))
    from syrinx_amd import SxqError
    with pytest.raises(SxqError) as e:
        lm.step(ids=torch.zeros((1, 11), dtype=torch.int32))
    assert "full" in str(e.value)


def _replay_all(ora, lm, cfg, W, lengths, step, frames, logits, hidden, what, split=False):
    """Op-by-op replay of one traced step of every stream (projections bit-exact, or with
    split the O and down projections to _split_close; glue to GLUE_RTOL), the step's logits
    and hidden against it, and the greedy argmax."""
    tr = lm.trace(len(lengths))
    got = logits.cpu().numpy()
    for s_ in range(len(lengths)):
        want = _replay_step(ora, lm, cfg, W, tr, s_, lengths[s_] + step, frame=frames[s_], split=split)
        _bits_equal(got[s_], want, f"{what} stream {s_} head projection")
        _bits_equal(hidden.cpu().numpy()[s_], tr["final_hn"][s_], f"{what} stream {s_} hidden")


@pytest.mark.parametrize("mode", ["split", "exact"])
def test_sixteen_streams_ragged_kv_256_to_2048(cuda, ora, model_oracle, monkeypatch, mode):
    """The skinny-batch configuration: 16 streams at the Qwen3-4B width (two layers, a
    4096-row head), KV lengths drawn uniformly from 256..2048: 16-row matrix-core GEMVs,
    16-stream fused attention with many splits per stream, the 16-stream argmax.  Two
    consecutive steps, each replayed op by op for every stream (projections bit-exact,
    the appended K/V rows checked, so the second step also verifies what the first
    wrote), and each compared end to end with the per-stream oracle model.  At this
    width nearly every step has an activation within 1e-5 of a Q8 rounding tie, so the
    end-to-end comparison is held to the flip bound only; the replay is the exact check.
    "split": the engine's default, whose O and down projections (160 tiles of 16 rows)
    split K over workgroups, held to 1e-6 * sum |w x| per output; "exact":
    SXQ_BIT_EXACT=1, every projection bit-identical to the oracle."""
    if mode == "exact":
        monkeypatch.setenv("SXQ_BIT_EXACT", "1")  # read at each launch (captured with the graph)
    import random
    r = random.Random(5)
    lengths = [r.randint(256, 2048) for _ in range(16)]
    cfg = D.fish_s2_slow_ar_config(n_layers=2, max_seq=2048 + 8, max_batch=16, vocab=4096, n_codebooks=10,
                                   codebook_size=64, semantic_begin=3000, semantic_end=4095)
    lm, W = _build_dev(cfg, cuda, 31)
    orc = model_oracle.OracleDecoder(cfg, W, 16)
    _prefill(lm, orc, cfg, lengths, seed=32)
    lm.enable_trace()
    rng = np.random.default_rng(33)
    for step in range(2):
        fr = _frames(rng, 16, cfg)
        logits, nxt, hidden = lm.step(ids=torch.from_numpy(fr), graph=True, want_hidden=True)
        _replay_all(ora, lm, cfg, W, lengths, step, list(fr), logits, hidden, f"16 streams step {step}",
                    split=mode == "split")
        got = logits.cpu().numpy()
        assert (nxt.cpu().numpy() == got.argmax(1)).all()
        for s_ in range(16):
            _check(got[s_], orc, orc.step_one(s_, frame=fr[s_]), f"16 streams step {step} stream {s_} "
                                                                   f"(len {lengths[s_] + step})")
    assert lm.lengths(16) == [L + 2 for L in lengths]


def test_split_k_gemv_step_is_deterministic(cuda):
    """The 16-row GEMVs with K split over workgroups add the slices' chains in a fixed
    order whichever slice finishes last: the same step (9 ragged streams, the Qwen3-4B
    width, graph-replayed and eager) gives the same bits on every run."""
    cfg = _fish_small(n_layers=2, max_batch=9)
    lengths = [5, 70, 17, 0, 33, 1, 48, 60, 9]
    fr = _frames(np.random.default_rng(47), 9, cfg)
    outs = []
    for graph in (True, True, False):
        lm, _ = _build_dev(cfg, cuda, 45)
        lm.kv_fill_random(lengths, seed=46)
        for _ in range(3):
            lm.set_lengths(lengths)
            logits, _, hidden = lm.step(ids=torch.from_numpy(fr), graph=graph, want_hidden=True)
            outs.append((logits.cpu().numpy(), hidden.cpu().numpy()))
        del lm
    for i, (lg, hd) in enumerate(outs[1:], 1):
        _bits_equal(lg, outs[0][0], f"run {i}: logits")
        _bits_equal(hd, outs[0][1], f"run {i}: hidden")


@pytest.mark.parametrize("width", [2560, 1024])
def test_persistent_matrix_core_gemv_grids_agree(cuda, monkeypatch, width):
    """The 5..16-row matrix-core GEMV with each workgroup walking many 16-row tiles (grid
    targets of 3 and 7 workgroups: the chunk pipeline runs across tile boundaries, chunk
    counts 1, 3, 4 and 10, partial last tiles) gives the bits of one workgroup per tile:
    logits and hidden state of one step of 9 ragged streams through every projection
    (wqkv, wo, w1|w3, w2, head) at the Qwen3-4B width and at a 1024-wide model."""
    kw = {} if width == 2560 else dict(dim=1024, n_heads=8, n_kv_heads=2, intermediate=2816)
    cfg = _fish_small(n_layers=1, max_batch=9, **kw)
    lengths = [5, 70, 17, 0, 33, 1, 48, 60, 9]
    fr = _frames(np.random.default_rng(43), 9, cfg)
    outs = []
    for target in ("0", "3", "7"):
        monkeypatch.setenv("SXQ_GEMV_REC_WG", target)
        lm, _ = _build_dev(cfg, cuda, 41)
        lm.kv_fill_random(lengths, seed=42)
        logits, _, hidden = lm.step(ids=torch.from_numpy(fr), want_hidden=True)
        outs.append((logits.cpu().numpy(), hidden.cpu().numpy()))
        del lm
    for target, (lg, hd) in zip(("3", "7"), outs[1:]):
        _bits_equal(lg, outs[0][0], f"width {width}, {target} workgroups: logits")
        _bits_equal(hd, outs[0][1], f"width {width}, {target} workgroups: hidden")


def test_cosyvoice2_q8_0_24_layers_at_kv_512(cuda, ora, model_oracle):
    """CosyVoice2 LM at its configuration: 24 layers, Q8_0, KV prefilled to 512
    positions (eight 64-position attention splits at head_dim 64).  Two steps (an
    embedding input, then a token id through the speech-embedding table), each
    replayed op by op and compared end to end with the oracle model (flip bound)."""
    cfg = D.cosyvoice2_lm_config(n_layers=24, max_seq=520, dtype=GgmlDType.Q8_0)
    lm, W = _build_dev(cfg, cuda, 34)
    orc = model_oracle.OracleDecoder(cfg, W, 1)
    _prefill(lm, orc, cfg, [512], seed=35)
    lm.enable_trace()
    rng = np.random.default_rng(36)
    emb = rng.standard_normal((1, cfg.dim)).astype(np.float32)
    logits, _, hidden = lm.step(embeds=torch.from_numpy(emb), graph=True, want_hidden=True)
    _replay_all(ora, lm, cfg, W, [512], 0, [None], logits, hidden, "cv2 kv512 step 0")
    _check(logits.cpu().numpy()[0], orc, orc.step_one(0, embed=emb[0]), "cv2 kv512 step 0")
    tok = np.array([[4321]], np.int32)
    logits, _, hidden = lm.step(ids=torch.from_numpy(tok), graph=True, want_hidden=True)
    _replay_all(ora, lm, cfg, W, [512], 1, list(tok), logits, hidden, "cv2 kv512 step 1")
    _check(logits.cpu().numpy()[0], orc, orc.step_one(0, frame=tok[0]), "cv2 kv512 step 1")
    assert lm.lengths(1) == [514]


def _fork(orc):
    """A copy of an oracle decoder that shares its weights and owns its caches."""
    import copy
    o2 = copy.copy(orc)
    o2.k = copy.deepcopy(orc.k)
    o2.v = copy.deepcopy(orc.v)
    return o2


@pytest.mark.parametrize("dtype", [GgmlDType.Q4K, GgmlDType.Q8_0])
def test_full_36_layer_step_at_kv_1024(cuda, ora, model_oracle, dtype):
    """The headline model at full size: 36 layers, the full 155776-row tied head, KV
    1024, every projection Q4_K -- and the same model with Q8_0 projections (the decode
    configuration's second weight format: 4.28 GB per token, a 424 MB head).  One step
    replayed op by op over all 36 layers (every projection and the head bit-exact).  End
    to end, Q8 rounding-tie flips compound over 36 layers, so the bound is the oracle's
    own sensitivity: the same oracle step on an embedding perturbed by 2^-21 relative
    (about the size of the glue ops' float differences) moves the logits by d_ref, and
    the GPU must stay within LOGIT_RTOL_FLIP + 2 d_ref."""
    cfg = D.fish_s2_slow_ar_config(n_layers=36, max_seq=1032, max_batch=1, dtype=dtype)
    lm, W = _build_dev(cfg, cuda, 37)
    orc = model_oracle.OracleDecoder(cfg, W, 1)
    _prefill(lm, orc, cfg, [1024], seed=38)
    lm.enable_trace()
    fr = _frames(np.random.default_rng(39), 1, cfg)
    logits, nxt, hidden = lm.step(ids=torch.from_numpy(fr), graph=True, want_hidden=True)
    _replay_all(ora, lm, cfg, W, [1024], 0, list(fr), logits, hidden, "qwen3-4b 36 layers")
    got = logits.cpu().numpy()[0]
    assert int(nxt[0]) == int(np.argmax(got))
    refs = []
    for sign in (1.0, -1.0):
        o2 = _fork(orc)
        emb = o2.embed(fr[0]) * np.float32(1.0 + sign * 2.0 ** -21)
        refs.append(o2.step_one(0, embed=emb.astype(np.float32)))
    want = orc.step_one(0, frame=fr[0])
    d_ref = max(_rel(r_, want) for r_ in refs)
    err = _rel(got, want)
    print(f"qwen3-4b 36 layers: rel err {err:.2e}, oracle under a 2^-21 input perturbation {d_ref:.2e}")
    assert err <= LOGIT_RTOL_FLIP + 2.0 * d_ref, (err, d_ref)

def test_slow_step_returns_logits_and_hidden(cuda, ora):
    """SlowAr.slow_step returns (semantic_logits, hidden) as SlowAr::slow_step does
    (crates/syrinx-fish/src/s2/slow_ar.rs:259-271): hidden is the post-final-RMSNorm
    state [1, 1, dim] the head multiplies (slow_ar.rs:207-246)."""
    cfg = _fish_small()
    lm = D.SlowAr(cfg, device=cuda)
    lm.init_random(seed=44, std=0.02)
    lm.kv_fill_random([20], seed=45)
    lm.enable_trace()
    fr = _frames(np.random.default_rng(46), 1, cfg)[0]
    logits, hidden = lm.slow_step(fr, pos=20)
    assert logits.shape == (cfg.vocab,) and hidden.shape == (1, 1, cfg.dim)
    tr = lm.trace(1)
    _bits_equal(hidden.cpu().numpy()[0, 0], tr["final_hn"][0], "hidden == final RMSNorm output")
    h_last = tr["layers"][-1]["h_out"][0]
    _glue_close(hidden.cpu().numpy()[0, 0], ora.rms_norm(h_last, np.ones(cfg.dim, np.float32), cfg.norm_eps),
                "hidden vs oracle RMSNorm of the last residual")
    assert int(lm.last_argmax()[0]) == int(np.argmax(logits.cpu().numpy()))


# ----------------------------------------------------------------------------- prefill
def _f16_bound_ok(got, x, blocks, dt, k, what, bias=None):
    """A projection of the f16 MFMA prefill GEMM: within the f16 rounding bound of the
    f64 product of the exactly dequantized weight (the QMatMul GEMM's contract)."""
    import oracle as ora_mod
    wd = ora_mod.dequantize(dt, blocks, k).reshape(-1, k).astype(np.float64)
    y64 = x.astype(np.float64) @ wd.T + (0.0 if bias is None else bias.astype(np.float64))
    S = np.abs(x).astype(np.float64) @ np.abs(wd).T
    tol = (2.0 ** -10 + k * 2.0 ** -24) * S + 2.0 ** -24 * np.abs(x).sum(1, keepdims=True) + 2.0 ** -24 * np.abs(
        wd).sum(1)[None, :] + 1e-30
    err = np.abs(got.astype(np.float64) - y64)
    assert (err <= tol).all(), f"{what}: {(err > tol).sum()} beyond the f16 bound"


def _replay_prefill(ora, lm, cfg, W, tr, counts, lens0, frames, exact):
    """Check every op of a traced prefill: token t of stream s sits at position
    lens0[s] + i; projections bit-exact (exact / Q8_0 / Q4_0) or within the f16 bound (the
    Q4_K GEMM at >= 64 rows), glue to GLUE_RTOL, attention re-run by the oracle over the
    GPU's own cache (whose rows are checked against the traced keys and values)."""
    dt = int(cfg.weight_dtype)
    hd, nh, nkv = cfg.head_dim, cfg.n_heads, cfg.n_kv_heads
    G = nh // nkv
    T = sum(counts)
    gemm_f16 = dt == int(GgmlDType.Q4K) and not exact and T >= 64
    rows = [(s, lens0[s] + i) for s in range(len(counts)) for i in range(counts[s])]
    maxpos = max(p for _, p in rows) + 1
    cos, sin = (ora.rope_tables_interleaved(maxpos, hd, cfg.rope_theta) if cfg.rope_interleaved
                else ora.rope_tables_half(maxpos, hd, cfg.rope_theta))
    rope = ora.rope_interleaved if cfg.rope_interleaved else ora.rope_half
    if frames is not None:
        import model
        orc = model.OracleDecoder(cfg, W, 1)
        for t in range(T):
            _bits_equal(tr["embed"][t], orc.embed(frames[t]), f"embedding row {t}")

    def proj(x, key, what, bias=None, res=None):
        blocks = W[key]
        if gemm_f16:
            y = None  # compared against the traced output below
            return y
        y = ora.matmul(dt, x, blocks)
        if bias is not None:
            y = (y + bias[None, :]).astype(np.float32)
        if res is not None:
            y = (res + y).astype(np.float32)
        return y

    caches = {}
    for l, Tl in enumerate(tr["layers"]):
        h_in = tr["embed"] if l == 0 else tr["layers"][l - 1]["h_out"]
        tag = f"layer {l}"
        for t in range(T):
            _glue_close(Tl["hn_attn"][t], ora.rms_norm(h_in[t], W[("attn_norm", l)], cfg.norm_eps), f"{tag} row {t} RMSNorm")
        bias = W[("bqkv", l)] if cfg.qkv_bias else None
        if gemm_f16:
            _f16_bound_ok(Tl["qkv"], Tl["hn_attn"], W[("wqkv", l)], dt, cfg.dim, f"{tag} qkv", bias)
        else:
            _bits_equal(Tl["qkv"], proj(Tl["hn_attn"], ("wqkv", l), "qkv", bias), f"{tag} qkv projection")
        for t, (s, p) in enumerate(rows):
            q = Tl["qkv"][t][: nh * hd].reshape(nh, hd)
            k = Tl["qkv"][t][nh * hd:(nh + nkv) * hd].reshape(nkv, hd)
            v = Tl["qkv"][t][(nh + nkv) * hd:].reshape(nkv, hd)
            if cfg.qk_norm:
                q = np.stack([ora.rms_norm(q[i], W[("q_norm", l)], cfg.norm_eps) for i in range(nh)])
                k = np.stack([ora.rms_norm(k[i], W[("k_norm", l)], cfg.norm_eps) for i in range(nkv)])
            _glue_close(Tl["q"][t], rope(q, cos[p], sin[p]).reshape(-1), f"{tag} row {t} QK-norm + RoPE (q)")
            kr = rope(k, cos[p], sin[p])
            ctx = np.zeros(nh * hd, np.float32)
            for g in range(nkv):
                if (l, s, g) not in caches:
                    kc, vc = lm.read_kv(l, s, g, 0, lens0[s] + counts[s])
                    caches[(l, s, g)] = (kc.cpu().numpy(), vc.cpu().numpy())
                kc, vc = caches[(l, s, g)]
                _glue_close(kc[p], kr[g], f"{tag} row {t} key (head {g})")
                _bits_equal(vc[p], v[g], f"{tag} row {t} value (head {g})")
                for i in range(g * G, (g + 1) * G):
                    ctx[i * hd:(i + 1) * hd] = ora.attend_one(Tl["q"][t][i * hd:(i + 1) * hd], kc[:p + 1], vc[:p + 1])
            _glue_close(Tl["ctx"][t], ctx, f"{tag} row {t} causal attention")
        if gemm_f16:
            _f16_bound_ok(Tl["h_mid"] - h_in, Tl["ctx"], W[("wo", l)], dt, nh * hd, f"{tag} O projection")
        else:
            _bits_equal(Tl["h_mid"], proj(Tl["ctx"], ("wo", l), "wo", res=h_in), f"{tag} O projection + residual")
        for t in range(T):
            _glue_close(Tl["hn_ffn"][t], ora.rms_norm(Tl["h_mid"][t], W[("ffn_norm", l)], cfg.norm_eps),
                        f"{tag} row {t} FFN RMSNorm")
        I = cfg.intermediate
        if gemm_f16:
            _f16_bound_ok(Tl["gu"][:, :I], Tl["hn_ffn"], W[("w1", l)], dt, cfg.dim, f"{tag} gate")
            _f16_bound_ok(Tl["gu"][:, I:], Tl["hn_ffn"], W[("w3", l)], dt, cfg.dim, f"{tag} up")
        else:
            _bits_equal(Tl["gu"], np.concatenate([proj(Tl["hn_ffn"], ("w1", l), "w1"),
                                                  proj(Tl["hn_ffn"], ("w3", l), "w3")], axis=1), f"{tag} gate|up")
        for t in range(T):
            _glue_close(Tl["act"][t], ora.silu_mul(Tl["gu"][t][:I], Tl["gu"][t][I:]), f"{tag} row {t} SiLU*mul")
        if gemm_f16:
            _f16_bound_ok(Tl["h_out"] - Tl["h_mid"], Tl["act"], W[("w2", l)], dt, I, f"{tag} down projection")
        else:
            _bits_equal(Tl["h_out"], proj(Tl["act"], ("w2", l), "w2", res=Tl["h_mid"]), f"{tag} down + residual")
    return rows


PREFILL_KINDS = {
    # name: (config, per-stream (cached length before, prompt tokens), exact)
    "fish_q4k_exact_1stream": (lambda: _fish_small(n_layers=2), [(0, 37)], True),
    # the RMSNorm quantizer by rows (128 and more), Q8_K, a dim of 2.5 passes of its workgroup
    "fish_q4k_exact_129_rows": (lambda: D.fish_s2_slow_ar_config(n_layers=1, max_seq=136, vocab=4096, n_codebooks=10,
                                                                 codebook_size=64, semantic_begin=3000,
                                                                 semantic_end=4095, intermediate=512), [(3, 129)], True),
    "fish_q4k_gemm_after_cache": (lambda: _fish_small(n_layers=1), [(20, 70)], False),
    "fish_q8_0_ragged3": (lambda: _fish_small(n_layers=2, max_batch=3, dtype=GgmlDType.Q8_0), [(5, 17), (0, 1),
                                                                                                (31, 40)], True),
    "cv2_q8_0_embeds": (lambda: D.cosyvoice2_lm_config(n_layers=2, max_seq=96, dtype=GgmlDType.Q8_0), [(9, 30)], True),
    "cv2_q4_0_gemm_rows": (lambda: D.cosyvoice2_lm_config(n_layers=1, max_seq=200, dtype=GgmlDType.Q4_0),
                           [(0, 130)], True),
    # the 512-token prompt of the prefill configuration at the Qwen3-4B width (one layer,
    # a 4096-row head): every projection on the f16 MFMA GEMM with its split plans
    "qwen3_4b_512_tokens": (lambda: D.fish_s2_slow_ar_config(n_layers=1, max_seq=520, vocab=4096, n_codebooks=10,
                                                             codebook_size=64, semantic_begin=3000,
                                                             semantic_end=4095), [(0, 512)], False),
}


@pytest.mark.parametrize("kind", list(PREFILL_KINDS))
def test_prefill_every_op_matches_oracle(cuda, ora, kind):
    """sxq_lm_prefill (SlowAr::prefill / prefill_batch, the CosyVoice2 prompt forward)
    replayed op by op over every prompt row, then the head on each stream's last row."""
    make, plan, exact = PREFILL_KINDS[kind]
    cfg = make()
    n = len(plan)
    lm, W = _build(cfg, cuda, 51, n)
    lens0 = [p[0] for p in plan]
    counts = [p[1] for p in plan]
    lm.kv_fill_random(lens0, seed=52)
    rng = np.random.default_rng(53)
    if kind.startswith("cv2"):
        embs = [rng.standard_normal((c, cfg.dim)).astype(np.float32) for c in counts]
        logits, nxt, hidden, tr = lm.prefill(embeds=[torch.from_numpy(e) for e in embs], exact=exact, trace=True)
        frames = None
    else:
        prompts = [_frames(rng, c, cfg) for c in counts]
        logits, nxt, hidden, tr = lm.prefill(prompts=[torch.from_numpy(p) for p in prompts], exact=exact, trace=True)
        frames = np.concatenate(prompts)
    _replay_prefill(ora, lm, cfg, W, tr, counts, lens0, frames, exact)
    last_h = tr["layers"][-1]["h_out"]
    got = logits.cpu().numpy()
    ends = np.cumsum(counts) - 1
    dt = int(cfg.weight_dtype)
    for s in range(n):
        _glue_close(tr["final_hn"][s], ora.rms_norm(last_h[ends[s]], W["final_norm"], cfg.norm_eps),
                    f"stream {s} final RMSNorm")
        _bits_equal(hidden.cpu().numpy()[s], tr["final_hn"][s], f"stream {s} hidden")
        want = ora.matmul(dt, tr["final_hn"][s][None], W["head"])[0]
        if cfg.head_bias:
            want = (want + W["head_bias"]).astype(np.float32)
        _bits_equal(got[s], want, f"stream {s} head")
        assert int(nxt[s]) == int(np.argmax(got[s]))
    assert lm.lengths(n) == [a + b for a, b in plan]


def test_prefill_then_decode_matches_oracle_model(cuda, model_oracle):
    """Prefill two ragged prompts, then decode two steps: every step's logits against the
    oracle model that ran the same tokens one at a time (flip bound end to end; the
    op-level replay above is the exact check)."""
    cfg = _fish_small(n_layers=2, max_batch=2)
    lm, W = _build(cfg, cuda, 54, 2)
    orc = model_oracle.OracleDecoder(cfg, W, 2)
    rng = np.random.default_rng(55)
    prompts = [_frames(rng, 23, cfg), _frames(rng, 9, cfg)]
    logits, nxt, hidden = lm.prefill(prompts=[torch.from_numpy(p) for p in prompts], exact=True)
    for s, p in enumerate(prompts):
        for i in range(len(p)):
            want = orc.step_one(s, frame=p[i])
        _check(logits.cpu().numpy()[s], orc, want, f"prefill stream {s} last position")
    for step in range(2):
        fr = _frames(rng, 2, cfg)
        lg, _ = lm.step(ids=torch.from_numpy(fr), graph=True)
        for s in range(2):
            _check(lg.cpu().numpy()[s], orc, orc.step_one(s, frame=fr[s]), f"decode after prefill {step} stream {s}")
    assert lm.lengths(2) == [25, 11]


def test_slow_ar_prefill_and_qwen2_all_logits_shapes(cuda, model_oracle):
    """SlowAr.prefill(prompt [1 + num_codebooks, T]) -> (logits [vocab], hidden [1, 1, dim])
    (slow_ar.rs:250-256); prefill_batch -> ([n, vocab], [n, 1, dim]); Qwen2Lm's
    forward_logits_cached over t_new > 1 embeddings returns every position's logits
    [b, t_new, vocab] (cv2/mod.rs:283-286), each against the oracle model."""
    cfg = _fish_small(n_layers=1, max_batch=2)
    lm = D.SlowAr(cfg, device=cuda)
    lm.init_random(seed=56)
    prompt = _frames(np.random.default_rng(57), 12, cfg).T  # [1 + num_codebooks, T]
    logits, hidden = lm.prefill(prompt)
    assert logits.shape == (cfg.vocab,) and hidden.shape == (1, 1, cfg.dim)
    assert lm.lengths(1) == [12]
    lm.reset()
    lb, hb = lm.prefill_batch([prompt, prompt[:, :5]])
    assert lb.shape == (2, cfg.vocab) and hb.shape == (2, 1, cfg.dim)
    np.testing.assert_array_equal(lb.cpu().numpy()[0], logits.cpu().numpy())
    assert lm.lengths(2) == [12, 5]

    cv = D.cosyvoice2_lm_config(n_layers=2, max_seq=64, dtype=GgmlDType.Q8_0)
    q2, W = _build(cv, cuda, 58, 1)
    orc = model_oracle.OracleDecoder(cv, W, 1)
    emb = np.random.default_rng(59).standard_normal((1, 6, cv.dim)).astype(np.float32)
    out = D.Qwen2Lm.forward_logits_cached(q2, torch.from_numpy(emb))
    assert out.shape == (1, 6, cv.vocab)
    for i in range(6):
        _check(out.cpu().numpy()[0, i], orc, orc.step_one(0, embed=emb[0, i]), f"cv2 prompt position {i}")


def test_prefill_argument_errors(cuda):
    cfg = _fish_small(n_layers=1, max_batch=2)
    cfg.max_seq = 16
    lm = D.DecoderLM(cfg, device=cuda)
    lm.init_random(seed=60)
    from syrinx_amd import SxqError
    with pytest.raises(SxqError, match="exceed"):
        lm.prefill(prompts=[np.zeros((17, 11), np.int32)])
    with pytest.raises(SxqError, match="no tokens"):
        lm.prefill(prompts=[np.zeros((3, 11), np.int32), np.zeros((0, 11), np.int32)])
    assert lm.lengths(2) == [0, 0]
