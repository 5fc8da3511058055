"""GPU kernels at the edges of their tiles: remainders, unaligned pointers, the smallest and
largest sizes each dispatch rule sends to them, against the CPU oracle."""
import ctypes

import numpy as np
import pytest
import torch

from syrinx_amd import GgmlDType, QMatMul, QTensor
from syrinx_amd._lib import BF16_INPUT, ERR_INVALID, SxqError, check, lib

pytestmark = pytest.mark.gpu

G = GgmlDType
G_Q8 = GgmlDType.Q8_0


@pytest.fixture(scope="module")
def cuda():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm GPU (torch.cuda.is_available() is False)")
    return torch.device("cuda:0")


def _rows(n, k, seed):
    """Normal rows with halves of zeros, of one value (ties), tiny and huge values."""
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    for i, v in enumerate((0.0, 0.5, 1e-30, 1e30)):
        x[i % n, : k // 2] = v if i < 2 else x[i % n, : k // 2] * v
    return x


@pytest.mark.parametrize("dt,k", [(G.Q8_0, 32), (G.Q8_0, 896), (G.Q4_0, 32), (G.Q4_0, 320), (G.Q4K, 256), (G.Q4K, 2560)])
@pytest.mark.parametrize("n", [1, 5, 33])
@pytest.mark.parametrize("shift", [0, 1])
def test_quantize_rows_remainders_and_unaligned(cuda, ora, dt, k, n, shift):
    """Block counts that do not fill a workgroup; x off 16-byte and out off 2-byte alignment."""
    x = _rows(n, k, 3 + n)
    nbytes = n * (k // dt.block_size()) * dt.type_size()
    xs = torch.zeros(n * k + 1, dtype=torch.float32, device=cuda)
    xs[shift: shift + n * k] = torch.from_numpy(x).to(cuda).reshape(-1)
    out = torch.full((nbytes + 2,), 0xA5, dtype=torch.uint8, device=cuda)
    check(lib().sxq_quantize_rows(0, int(dt), ctypes.c_void_p(xs.data_ptr() + 4 * shift), n, k,
                                  ctypes.c_void_p(out.data_ptr() + shift), torch.cuda.current_stream().cuda_stream))
    got = out.cpu().numpy()
    want = ora.quantize(int(dt), x).reshape(-1)
    np.testing.assert_array_equal(got[shift: shift + nbytes], want)
    assert (got[:shift] == 0xA5).all() and (got[shift + nbytes:] == 0xA5).all()


def _special_blocks():
    """[P, 256]: one special pattern each in one of the eight 32-element (sub-)blocks of an otherwise
    normal row -- infinities and NaN at the first, inner and last lanes of a block, alone, mixed,
    and over whole blocks and rows; ties of the largest magnitude with either sign first; the
    largest and subnormal floats; signed zeros."""
    inf, nan, big = np.float32(np.inf), np.float32(np.nan), np.finfo(np.float32).max
    pats = [{at: v} for v in (inf, -inf, nan, -nan, big, -big) for at in (0, 5, 31)]
    pats += [{i: v for i in range(32)} for v in (inf, -inf, nan, big, np.float32(1e-40), np.float32(0.0), np.float32(-0.0))]
    pats += [{3: inf, 20: -inf}, {20: inf, 3: -inf}, {0: nan, 31: inf}, {31: nan, 0: -inf}, {0: big, 31: -big},
             {9: 2.0, 2: -2.0}, {9: -2.0, 2: 2.0}, {17: 2.0, 16: -2.0}, {30: 2.0, 1: nan, 4: -2.0}, {7: np.float32(1e-40)},
             {i: np.float32(-0.0) if i % 3 else np.float32(0.0) for i in range(32)}]
    x = (np.random.default_rng(11).standard_normal((len(pats) + 3, 256)) * 0.02).astype(np.float32)
    for p, pat in enumerate(pats):
        for at, v in pat.items():
            x[p, 32 * (p % 8) + at] = v
    x[-3], x[-2] = nan, inf
    x[-1, ::7] = nan
    return x


@pytest.mark.parametrize("dt", [G.Q8_0, G.Q4_0, G.Q4K])
def test_quantize_infinities_nan_and_ties(cuda, ora, dt):
    """The oracle's bytes where a value is not finite or a maximum is tied."""
    x = _special_blocks()
    got = QTensor.quantize(torch.from_numpy(x).to(cuda), dt).data().cpu().numpy().reshape(len(x), -1)
    want = ora.quantize(int(dt), x).reshape(len(x), -1)
    bad = [int(r) for r in np.flatnonzero((got != want).any(1))]
    assert not bad, f"rows {bad}: {[(got[r][got[r] != want[r]][:4], want[r][got[r] != want[r]][:4]) for r in bad[:3]]}"


# (n, k, m): weight and row tiles of 16 / 32 / 64 rows with remainders,
# block counts below, at and past a chunk (4, 8, 16, 32 blocks)
Q80_SHAPES = [(1, 32, 5), (17, 320, 16), (16, 1024, 17), (130, 1056, 33), (896, 4864, 8), (77, 992, 64), (200, 160, 65),
              (1152, 896, 226), (2048, 1024, 500), (4100, 96, 130), (896, 4864, 226), (9728, 896, 50), (64, 2080, 300),
              # 32 x 32 tiles whose last row tile and weight tile hold one row: 1, 10 and 28 blocks
              (2049, 32, 97), (2049, 320, 97), (1153, 896, 225),
              # 400 tiles of 64 x 64 and more: remainders of rows, weight rows and blocks (3, 29, 5)
              (6565, 96, 257), (6564, 928, 226), (25700, 160, 33),
              # the lines of the dispatch: one 32-row tile of a wide weight, 16 rows of 513 tiles, 17 rows of
              # 514, a long K over few outputs (the GEMV up to 512 outputs and eight rows)
              (25700, 160, 32), (8200, 96, 9), (4112, 96, 17), (512, 8192, 6), (40, 7168, 8), (513, 7168, 5), (40, 7168, 9)]


@pytest.mark.parametrize("dt", [G.Q8_0, G.Q4_0])
@pytest.mark.parametrize("n,k,m", Q80_SHAPES)
def test_q80_matrix_core_bit_exact(cuda, ora, dt, n, k, m):
    """Five rows and more of Q8_0 / Q4_0: Candle's bits, with a bias and zero / tied rows."""
    rng = np.random.default_rng(n + k + m)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    w[0] = 0.0
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[1] = 0.0
    x[2, :32] = -3.0
    b = rng.standard_normal(n).astype(np.float32)
    blocks = ora.quantize(int(dt), w)
    qmm = QMatMul.from_qtensor(QTensor.from_blocks(blocks, (n, k), dt, device=cuda))
    got = qmm.forward(torch.from_numpy(x).to(cuda), bias=torch.from_numpy(b).to(cuda)).cpu().numpy()
    want = (ora.matmul(int(dt), x, blocks) + b[None, :]).astype(np.float32)
    assert (got == want).all(), f"{int((got != want).sum())} of {got.size} outputs differ"


@pytest.mark.parametrize("n,k,m", [(7, 256, 17), (40, 1536, 33), (1003, 2560, 63), (6144, 512, 48), (130, 1024, 21),
                                   # one to three rows past the last slab, around the widths from which they run alone
                                   (8170, 512, 17), (8177, 512, 33), (12270, 256, 18), (12280, 256, 50), (16360, 256, 19),
                                   (16370, 256, 35)])
def test_q4k_slabs_bit_exact(cuda, ora, n, k, m):
    """17..63 rows of Q4_K (and any count with exact=True): every 16-row slab of one launch, a
    partial last slab, weight tiles that are no multiple of eight."""
    rng = np.random.default_rng(n + k + m)
    w = (rng.standard_normal((n, k)) * 0.02).astype(np.float32)
    x = rng.standard_normal((m + 100, k)).astype(np.float32)
    b = rng.standard_normal(n).astype(np.float32)
    blocks = ora.quantize(ora.Q4K, w)
    qmm = QMatMul.from_qtensor(QTensor.from_blocks(blocks, (n, k), G.Q4K, device=cuda))
    want = (ora.matmul(ora.Q4K, x, blocks) + b[None, :]).astype(np.float32)
    bias = torch.from_numpy(b).to(cuda)
    assert (qmm.forward(torch.from_numpy(x[:m]).to(cuda), bias=bias).cpu().numpy() == want[:m]).all()
    assert (qmm.forward(torch.from_numpy(x).to(cuda), bias=bias, exact=True).cpu().numpy() == want).all()


@pytest.mark.parametrize("dt,k", [(G.Q4K, 512), (G.Q8_0, 96), (G.Q4_0, 320)])
@pytest.mark.parametrize("m", [2, 7, 40])
def test_bf16_rows_quantized_directly(cuda, dt, k, m):
    """bf16 x through the quantizer equals the f32 x of the same values, bit for bit, also from
    a base that is not 8-byte aligned."""
    g = torch.Generator(device=cuda).manual_seed(k + m)
    qmm = QMatMul.from_qtensor(QTensor.quantize(torch.randn(100, k, generator=g, device=cuda) * 0.02, dt))
    buf = torch.randn(m * k + 1, generator=g, device=cuda).bfloat16()
    for x in (buf[:-1].view(m, k), buf[1:].view(m, k)):
        assert torch.equal(qmm.forward(x), qmm.forward(x.float()))


@pytest.mark.parametrize("hd,G,nkv", [(128, 4, 2), (64, 7, 2), (128, 1, 2), (64, 64, 1), (128, 5, 1), (64, 64, 2)])
def test_prefill_attention_tiles(cuda, hd, G, nkv):
    """Causal attention of ragged prompts on top of filled caches against 64 bits: prompts of one
    token, of a partial and of several row tiles, caches that end inside a key tile."""
    from syrinx_amd.decoder import DecoderConfig, DecoderLM
    cfg = DecoderConfig(n_layers=1, dim=256, n_heads=G * nkv, n_kv_heads=nkv, head_dim=hd, intermediate=256, vocab=64,
                        max_seq=330, max_batch=4, weight_dtype=int(G_Q8), tied_embedding=0, qk_norm=0)
    lm = DecoderLM(cfg, device=cuda)
    lm.init_random(seed=5, std=0.05)
    gen = torch.Generator(device=cuda).manual_seed(hd + G)
    for counts in ([1, 31, 64, 130], [70, 33, 1, 65]):  # the second call starts at the first's lengths
        pos0 = lm.lengths(4)
        xs = [torch.randn(c, cfg.dim, generator=gen, device=cuda) * 3 for c in counts]
        logits, _, _, tr = lm.prefill(embeds=xs, all_logits=True, trace=True)
        tr = tr["layers"][0]
        if pos0[0] == 0:
            first = xs, logits
        q = torch.from_numpy(tr["q"]).to(cuda).double().view(-1, G * nkv, hd)
        got = torch.from_numpy(tr["ctx"]).to(cuda).double().view(-1, G * nkv, hd)
        at = 0
        for s, c in enumerate(counts):
            for g in range(nkv):
                k, v = (t.double() for t in lm.read_kv(0, s, g, 0, pos0[s] + c))
                mask = torch.arange(pos0[s] + c, device=cuda)[None, :] > pos0[s] + torch.arange(c, device=cuda)[:, None]
                for h in range(G):
                    sc = (q[at:at + c, g * G + h] @ k.t() / hd ** 0.5).masked_fill(mask, float("-inf"))
                    want = torch.softmax(sc, -1) @ v
                    # f32 scores of magnitude |s| err by ~|s| 2^-24 sqrt(hd), which the exponential
                    # passes on to the weights; the weighted sum errs by about as much again
                    tol = 8 * 2.0 ** -24 * (sc[~mask].abs().max() + 4) * hd ** 0.5 * v.abs().max()
                    err = (got[at:at + c, g * G + h] - want).abs().max()
                    assert err <= tol, f"counts {counts} stream {s} head {g * G + h}: {float(err):.3g} > {float(tol):.3g}"
            at += c
    lm.reset(4)  # without a trace the context goes to the O projection as blocks only
    assert torch.equal(lm.prefill(embeds=first[0], all_logits=True)[0], first[1])


@pytest.mark.parametrize("dt,k", [(G.Q4K, 512), (G.Q8_0, 896), (G.Q4_0, 320)])
@pytest.mark.parametrize("m", [1, 5, 70])
def test_forward_workspaces(cuda, dt, k, m):
    """The forward's workspace per call: calls that alternate between streams, and a captured
    call replayed between eager ones (one row of Q8_0 / Q4_0 needs no workspace)."""
    gen = torch.Generator(device=cuda).manual_seed(k + m)
    qmm = QMatMul.from_qtensor(QTensor.quantize(torch.randn(300, k, generator=gen, device=cuda) * 0.02, dt))
    xs = [torch.randn(m, k, generator=gen, device=cuda) for _ in range(8)]
    want = [qmm.forward(x).clone() for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(device=cuda) for _ in range(2)]
    got = []
    for i, x in enumerate(xs):
        with torch.cuda.stream(streams[i % 2]):
            got.append(qmm.forward(x))
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    xin = xs[0].clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = qmm.forward(xin)
    for x, w in zip(xs[:4], want):
        xin.copy_(x)
        graph.replay()
        eager = qmm.forward(xs[5])
        torch.cuda.synchronize()
        assert torch.equal(y, w) and torch.equal(eager, want[5])


def test_row_limit_is_the_librarys(cuda):
    qmm = QMatMul.from_qtensor(QTensor.quantize(torch.ones(1, 32, device=cuda), G.Q8_0))
    assert qmm.forward(torch.zeros(65535, 32, device=cuda)).shape == (65535, 1)
    with pytest.raises(SxqError, match="65536 rows exceed the 65535-row limit"):
        qmm.forward(torch.zeros(2, 32768, 32, device=cuda))


@pytest.mark.parametrize("dt,k", [(G.Q4K, 512), (G.Q8_0, 896), (G.Q4_0, 320)])
@pytest.mark.parametrize("m", [1, 2])
@pytest.mark.parametrize("bf16", [False, True])
def test_queried_workspace_is_enough(cuda, dt, k, m, bf16):
    """The C sequence of a caller with its own memory: query the size, allocate that many bytes
    (a null pointer for none), run; one byte less is refused where any is needed."""
    gen = torch.Generator(device=cuda).manual_seed(k + m)
    qmm = QMatMul.from_qtensor(QTensor.quantize(torch.randn(300, k, generator=gen, device=cuda) * 0.02, dt))
    x = torch.randn(m, k, generator=gen, device=cuda)
    x = x.bfloat16() if bf16 else x
    flags = BF16_INPUT if bf16 else 0
    need = ctypes.c_size_t()
    check(lib().sxq_qmm_workspace_size(qmm._h, m, flags, ctypes.byref(need)))
    assert need.value > 0 or (m == 1 and dt != G.Q4K and not bf16)
    ws = torch.empty(need.value, dtype=torch.uint8, device=cuda)
    y = torch.zeros(m, 300, device=cuda)

    def run(nbytes):
        return lib().sxq_qmm_forward_ws(qmm._h, ctypes.c_void_p(x.data_ptr()), (ctypes.c_int64 * 2)(m, k), 2, None,
                                        ctypes.c_void_p(y.data_ptr()), None, flags,
                                        ctypes.c_void_p(ws.data_ptr() if nbytes else None), nbytes,
                                        torch.cuda.current_stream().cuda_stream)

    check(run(need.value))
    assert torch.equal(y, qmm.forward(x))
    if need.value:
        assert run(need.value - 1) == ERR_INVALID and run(0) == ERR_INVALID


@pytest.mark.parametrize("dim,inter,T", [(256, 512, 64), (1280, 4352, 65), (4352, 256, 257)])
def test_prefill_f16_sources(cuda, dim, inter, T):
    """The f16 prompt path, whose projections prepare their operand from the RMSNorm and the
    SwiGLU: the rows a trace records against 64 bits, and the same logits without a trace."""
    from syrinx_amd.decoder import ATTN_NORM, FFN_NORM, DecoderConfig, DecoderLM
    cfg = DecoderConfig(n_layers=1, dim=dim, n_heads=4, n_kv_heads=2, head_dim=64, intermediate=inter, vocab=64,
                        max_seq=T, max_batch=1, weight_dtype=int(G.Q4K), tied_embedding=0, qk_norm=0)
    lm = DecoderLM(cfg, device=cuda)
    lm.init_random(seed=7, std=0.05)
    gen = torch.Generator(device=cuda).manual_seed(dim + T)
    w = {n: 1 + 0.2 * torch.randn(dim, generator=gen, device=cuda) for n in (ATTN_NORM, FFN_NORM)}
    for n, v in w.items():
        lm.set_vector(0, n, v)
    x = torch.randn(T, dim, generator=gen, device=cuda) * torch.logspace(-3, 3, T, device=cuda)[:, None]
    logits, _, hidden, tr = lm.prefill(embeds=[x], all_logits=True, trace=True)
    lm.reset(1)
    again = lm.prefill(embeds=[x], all_logits=True)
    assert torch.equal(again[0], logits) and torch.equal(again[2], hidden)
    layer = {k: torch.from_numpy(v).to(cuda).double().view(T, -1) for k, v in tr["layers"][0].items()}

    def norm(h, n):
        return h / (h.pow(2).mean(-1, keepdim=True) + cfg.norm_eps).sqrt() * w[n].double()

    gate, up = layer["gu"].split(inter, -1)
    for name, got, want in [("hn_attn", layer["hn_attn"], norm(x.double(), ATTN_NORM)),
                            ("hn_ffn", layer["hn_ffn"], norm(layer["h_mid"], FFN_NORM)),
                            ("act", layer["act"], torch.nn.functional.silu(gate) * up)]:
        # a few roundings of f32 (the sum of squares is a tree: its error grows with its depth)
        err = ((got - want).abs() / want.abs().clamp_min(1e-30)).max()
        assert err < 32 * 2.0 ** -24, f"{name}: relative error {float(err):.3g}"
