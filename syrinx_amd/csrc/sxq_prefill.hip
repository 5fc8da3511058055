// sxq_prefill.hip -- the glue of a prompt (many tokens per stream) through the decoder:
// per-token QK-RMSNorm + RoPE + KV-cache write, and causal GQA attention of the prompt's
// queries over each stream's cache.
//
// Reference: SlowAr::prefill / prefill_batch (crates/syrinx-fish/src/s2/slow_ar.rs:250-256,
// 404-454) and Qwen2Lm::forward_hidden_cached (crates/syrinx-lm/src/cv2/mod.rs:261-286):
// the new tokens sit at positions cache.len() .. cache.len() + t_new, each query attends
// its own stream's keys up to its own position (causal_mask_at, s2/nn.rs:208-218,
// cv2/attention.rs:120-141), scores (q . k) / sqrt(head_dim), softmax in f32.
#include "sxq_attn_dev.h"
#include "sxq_decoder.h"

namespace sxq {

// grid (T, n_heads + 2 * n_kv), one wave per head of token t's fused qkv row: the same
// per-head arithmetic (rope_load / rope_pair) as the fused decode attention, at the
// token's own stream and position (tok[t] = {stream, position}).
template <int HD>
__global__ __launch_bounds__(64) void k_prefill_rope_kv(const float* __restrict__ qkv, int qkv_n, int nh, int nkv,
                                                        const float* __restrict__ qn, const float* __restrict__ kn,
                                                        float eps, float inv_hd, int interleaved,
                                                        const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                                                        const int2* __restrict__ tok, float* __restrict__ qout,
                                                        float* __restrict__ kc, float* __restrict__ vc,
                                                        int64_t kv_stream_stride, int max_seq) {
    const int t = blockIdx.x, hid = blockIdx.y, lane = threadIdx.x;
    const int2 sp = tok[t];
    const int s = sp.x, pos = sp.y;
    const float* src = qkv + (int64_t)t * qkv_n + (int64_t)hid * HD;
    const bool is_q = hid < nh, is_k = !is_q && hid < nh + nkv;
    if (!is_q && !is_k) {  // V: stored as projected
        const int g = hid - nh - nkv;
        float* dst = vc + (int64_t)s * kv_stream_stride + ((int64_t)g * max_seq + pos) * HD;
        for (int d = lane; d < HD; d += 64) dst[d] = src[d];
        return;
    }
    float* dst = is_q ? qout + ((int64_t)t * nh + hid) * HD
                      : kc + (int64_t)s * kv_stream_stride + ((int64_t)(hid - nh) * max_seq + pos) * HD;
    const float* nw = is_q ? qn : kn;
    const RopeIn ri = rope_load<HD>(src, nw, interleaved, cos_t + (int64_t)pos * (HD / 2),
                                    sin_t + (int64_t)pos * (HD / 2), lane);
    rope_store<HD>(rope_pair<HD>(ri, nw != nullptr, eps, inv_hd, lane), interleaved, dst, nullptr, lane);
}

constexpr int kPfRows = 64;  // query rows (tokens x heads of one KV group) per workgroup
constexpr int kPfKeys = 64;  // key positions per LDS tile: 32 for each half of the waves

// LDS row strides (floats): a lane's float4 reads of 16 consecutive keys, and the value reads
// of 32 dims of two keys four apart, each hit every bank once.
constexpr int pf_kstride(int hd) { return hd + 4; }
constexpr int pf_vstride(int hd) { return hd + 8; }
size_t prefill_attn_lds(int hd) {
    const size_t tiles = sizeof(float) * (size_t)kPfKeys * (pf_kstride(hd) + pf_vstride(hd));
    const size_t merge = sizeof(float) * 2 * 64 * (size_t)(hd / 2 + 2);  // two waves' accumulators, m and l
    return tiles > merge ? tiles : merge;
}

typedef float v16f __attribute__((ext_vector_type(16)));

// One workgroup (256 threads) per (tile, KV group): a tile is up to kPfRows / G
// consecutive prompt tokens of one stream (tile = {stream, first token row t0, count,
// position p0 of token t0}); its rows are r = i * G + hh (token i, query head g * G + hh).
// Everything is f32 on the f32 matrix cores (v_mfma_f32_32x32x2_f32), transposed so that a
// row's softmax stays in its lane: wave w holds rows 32 (w & 1) .. +31 and takes the 32-key
// halves w >> 1 of the tiles; lane (c, h) = (lane & 31, lane >> 5) owns row c.
//   scores^T = K Q^T: result i of a lane is key 8 (i / 4) + 4 h + i % 4 of its row (the query
//     row is in the lane's registers for the whole kernel; K's dims are taken in the order 8 u
//     + 4 h + t, so that a lane reads float4s);
//   out^T += V^T P^T: the probabilities are already the operand the product needs (MFMA i takes
//     that key from half h), V comes from LDS a row of 32 dims at a time.
// Each wave keeps an online softmax (running max m, sum l, rescaled accumulator) over its own
// keys, masking keys past a row's own position; the two halves' results meet in LDS at the end.
// Bound by the f32 matrix cores (64 cycles per 4096 flops): 1412 ragged tokens of 32 / 8 heads of
// 128 in 196 us per layer, 226 tokens of 14 / 2 heads of 64 in 21.4 us; with the same tiles
// on the VALU (a score per thread, four threads per row) 591 and 66 us.  Tiles are taken last
// first: the last tokens of a prompt attend the most keys.
template <int HD>
__global__ __launch_bounds__(256, 2) void k_prefill_attn(const float* __restrict__ q, const float* __restrict__ kc,
                                                         const float* __restrict__ vc, const int4* __restrict__ tiles,
                                                         int nh, int nkv, int max_seq, int64_t kv_stream_stride,
                                                         float scale, float* __restrict__ ctx) {
    extern __shared__ float4 smem4[];
    constexpr int KS = pf_kstride(HD), VS = pf_vstride(HD), U = HD / 8, DG = HD / 32;
    const int4 tl = tiles[gridDim.x - 1 - blockIdx.x];
    const int s = tl.x, t0 = tl.y, cnt = tl.z, p0 = tl.w;
    const int g = blockIdx.y, G = nh / nkv, R = cnt * G;
    float* kt = (float*)smem4;      // [kPfKeys][KS]
    float* vt = kt + kPfKeys * KS;  // [kPfKeys][VS]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane & 31, h = lane >> 5, half = wave >> 1;
    const int row = 32 * (wave & 1) + c;
    const int rr = min(row, R - 1);  // rows past the tile compute on a copy and store nothing
    const int64_t qoff = (int64_t)(t0 + rr / G) * nh * HD + (g * G + rr % G) * HD;
    const int qpos = p0 + rr / G;
    float4 qv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) qv[u] = *(const float4*)(q + qoff + 8 * u + 4 * h);
    float m = -INFINITY, l = 0.0f;
    v16f o[DG];
#pragma unroll
    for (int d = 0; d < DG; ++d) o[d] = v16f{};
    const int64_t koff = (int64_t)s * kv_stream_stride + (int64_t)g * max_seq * HD;
    const int kend = p0 + cnt;
    for (int j0 = 0; j0 < kend; j0 += kPfKeys) {
        lds_barrier();  // the previous tile is no longer read
        for (int e = tid; e < kPfKeys * (HD / 4); e += 256) {
            const int key = e / (HD / 4), d = 4 * (e % (HD / 4));
            float4 kv = make_float4(0.f, 0.f, 0.f, 0.f), vv = kv;
            if (j0 + key < kend) {
                kv = *(const float4*)(kc + koff + (int64_t)(j0 + key) * HD + d);
                vv = *(const float4*)(vc + koff + (int64_t)(j0 + key) * HD + d);
            }
            *(float4*)(kt + key * KS + d) = kv;
            *(float4*)(vt + key * VS + d) = vv;
        }
        lds_barrier();
        const int jb = j0 + 32 * half;  // this wave's first key
        if (jb >= kend) continue;       // uniform per wave; every wave reaches each barrier
        v16f sc = v16f{};
        const float* kr = kt + (32 * half + c) * KS + 4 * h;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float4 kv = *(const float4*)(kr + 8 * u);
            sc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.x, qv[u].x, sc, 0, 0, 0);
            sc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.y, qv[u].y, sc, 0, 0, 0);
            sc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.z, qv[u].z, sc, 0, 0, 0);
            sc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.w, qv[u].w, sc, 0, 0, 0);
        }
        float bm = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int j = jb + 8 * (i >> 2) + 4 * h + (i & 3);
            sc[i] = j <= qpos ? sc[i] * scale + 0.0f : -INFINITY;
            bm = fmaxf(bm, sc[i]);
        }
        bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
        const float mn = fmaxf(m, bm);
        const float corr = mn == -INFINITY ? 1.0f : expf(m - mn);
        float ps = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            sc[i] = sc[i] == -INFINITY ? 0.0f : expf(sc[i] - mn);
            ps += sc[i];
        }
        ps += __shfl_xor(ps, 32, 64);
        l = l * corr + ps;
        m = mn;
        const float* vr = vt + (32 * half + 4 * h) * VS + c;
#pragma unroll
        for (int d = 0; d < DG; ++d) {
#pragma unroll
            for (int i = 0; i < 16; ++i) o[d][i] *= corr;
#pragma unroll
            for (int i = 0; i < 16; ++i)
                o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[(8 * (i >> 2) + (i & 3)) * VS + 32 * d], sc[i], o[d], 0, 0, 0);
        }
    }
    // the second half's waves hand their rows to the first half's
    lds_barrier();
    float* ex = (float*)smem4 + (wave & 1) * 64 * (HD / 2 + 2);
    if (half == 1) {
#pragma unroll
        for (int d = 0; d < DG; ++d)
#pragma unroll
            for (int i = 0; i < 16; ++i) ex[(16 * d + i) * 64 + lane] = o[d][i];
        ex[(HD / 2) * 64 + lane] = m;
        ex[(HD / 2 + 1) * 64 + lane] = l;
    }
    lds_barrier();
    if (half == 1 || row >= R) return;
    const float m1 = ex[(HD / 2) * 64 + lane], l1 = ex[(HD / 2 + 1) * 64 + lane];
    const float mn = fmaxf(m, m1);
    const float c0 = mn == -INFINITY ? 1.0f : expf(m - mn), c1 = mn == -INFINITY ? 1.0f : expf(m1 - mn);
    const float lt = l * c0 + l1 * c1;
#pragma unroll
    for (int d = 0; d < DG; ++d)
#pragma unroll
        for (int i = 0; i < 16; i += 4) {
            float v[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) v[t] = (o[d][i + t] * c0 + ex[(16 * d + i + t) * 64 + lane] * c1) / lt;
            *(float4*)(ctx + qoff + 32 * d + 2 * i + 4 * h) = make_float4(v[0], v[1], v[2], v[3]);
        }
}

// One thread per token t (and per tile index): stream-major order, stream s's tokens at
// rows base_s .. base_s + counts[s] - 1 and positions lens[s] .. lens[s] + counts[s] - 1.
__global__ __launch_bounds__(256) void k_prefill_tables(PrefillMeta pm, int T, int2* __restrict__ tok,
                                                        int4* __restrict__ tiles, int* __restrict__ last) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    int base = 0, tbase = 0;
    for (int s = 0; s < pm.n; ++s) {
        const int c = pm.counts[s], nt = (c + pm.tile_tokens - 1) / pm.tile_tokens;
        if (t >= base && t < base + c) tok[t] = make_int2(s, pm.lens[s] + (t - base));
        if (t >= tbase && t < tbase + nt) {
            const int i0 = (t - tbase) * pm.tile_tokens;
            tiles[t] = make_int4(s, base + i0, min(pm.tile_tokens, c - i0), pm.lens[s] + i0);
        }
        if (t == 0) last[s] = c > 0 ? base + c - 1 : -1;
        base += c;
        tbase += nt;
    }
    (void)T;
}

__global__ void k_prefill_advance(PrefillMeta pm, int* __restrict__ len) {
    const int s = threadIdx.x;
    if (s < pm.n) len[s] += pm.counts[s];
}

hipError_t launch_prefill_tables(const PrefillMeta& pm, int T, int* tok, int* tiles, int* last, hipStream_t s) {
    const int n_items = T + pm.n;  // tokens, and at most T + n tiles
    hipLaunchKernelGGL(k_prefill_tables, dim3((n_items + 255) / 256), dim3(256), 0, s, pm, T, (int2*)tok, (int4*)tiles,
                       last);
    return hipGetLastError();
}

hipError_t launch_prefill_advance(const PrefillMeta& pm, int* len, hipStream_t s) {
    hipLaunchKernelGGL(k_prefill_advance, dim3(1), dim3(64), 0, s, pm, len);
    return hipGetLastError();
}

// rows[i] = src[idx[i]] for n rows of `cols` floats (each stream's last prompt row).
__global__ __launch_bounds__(256) void k_gather_rows(const float* __restrict__ src, const int* __restrict__ idx,
                                                     int cols, float* __restrict__ dst) {
    const int i = blockIdx.x;
    const float* a = src + (int64_t)idx[i] * cols;
    for (int c = threadIdx.x; c < cols; c += 256) dst[(int64_t)i * cols + c] = a[c];
}

hipError_t launch_prefill_rope_kv(const float* qkv, int T, int qkv_n, int nh, int nkv, int hd, const float* qn,
                                  const float* kn, float eps, int interleaved, const float* cos_t, const float* sin_t,
                                  const int* tok, float* qout, float* kc, float* vc, int64_t kv_stream_stride,
                                  int max_seq, hipStream_t s) {
    if (hd != 64 && hd != 128) return hipErrorInvalidValue;
    const dim3 grid(T, nh + 2 * nkv);
    if (hd == 128)
        hipLaunchKernelGGL(k_prefill_rope_kv<128>, grid, dim3(64), 0, s, qkv, qkv_n, nh, nkv, qn, kn, eps,
                           1.0f / (float)hd, interleaved, cos_t, sin_t, (const int2*)tok, qout, kc, vc,
                           kv_stream_stride, max_seq);
    else
        hipLaunchKernelGGL(k_prefill_rope_kv<64>, grid, dim3(64), 0, s, qkv, qkv_n, nh, nkv, qn, kn, eps,
                           1.0f / (float)hd, interleaved, cos_t, sin_t, (const int2*)tok, qout, kc, vc,
                           kv_stream_stride, max_seq);
    return hipGetLastError();
}

bool prefill_attn_supported(int nh, int nkv, int hd) { return (hd == 64 || hd == 128) && nh / nkv <= kPfRows; }
int prefill_tile_tokens(int nh, int nkv) { return kPfRows / (nh / nkv); }

hipError_t launch_prefill_attn(const float* q, const float* kc, const float* vc, const int* tiles, int n_tiles, int nh,
                               int nkv, int hd, int max_seq, int64_t kv_stream_stride, float* ctx, hipStream_t s) {
    if (!prefill_attn_supported(nh, nkv, hd)) return hipErrorInvalidValue;
    if (n_tiles == 0) return hipSuccess;
    const size_t lds = prefill_attn_lds(hd);
    const float scale = (float)(1.0 / sqrt((double)hd));
    if (hd == 128) {
        static const hipError_t a = hipFuncSetAttribute((const void*)k_prefill_attn<128>,
                                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)prefill_attn_lds(128));
        if (a != hipSuccess) return a;
        hipLaunchKernelGGL(k_prefill_attn<128>, dim3(n_tiles, nkv), dim3(256), lds, s, q, kc, vc, (const int4*)tiles,
                           nh, nkv, max_seq, kv_stream_stride, scale, ctx);
    } else {
        static const hipError_t a = hipFuncSetAttribute((const void*)k_prefill_attn<64>,
                                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)prefill_attn_lds(64));
        if (a != hipSuccess) return a;
        hipLaunchKernelGGL(k_prefill_attn<64>, dim3(n_tiles, nkv), dim3(256), lds, s, q, kc, vc, (const int4*)tiles,
                           nh, nkv, max_seq, kv_stream_stride, scale, ctx);
    }
    return hipGetLastError();
}

hipError_t launch_gather_rows(const float* src, const int* idx, int n, int cols, float* dst, hipStream_t s) {
    hipLaunchKernelGGL(k_gather_rows, dim3(n), dim3(256), 0, s, src, idx, cols, dst);
    return hipGetLastError();
}

}  // namespace sxq
