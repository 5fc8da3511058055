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

constexpr int kPfRows = 64;  // query rows (tokens x heads of one KV group) per tile

typedef float v16f __attribute__((ext_vector_type(16)));

// Exchanges lanes 32..63 of a with lanes 0..31 of b.
SXQ_DEV void swap32(float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}
// Exchanges the odd 16-lane rows of a with the even ones of b (row 1 with 0, row 3 with 2).
SXQ_DEV void swap16(float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}

// A wave's share of a tile of ROWS rows of HD floats, straight to LDS: row r's 16-byte piece
// p goes to slot p ^ sw(r) of its row.  off(r) is the byte offset of row r's data.
template <int HD, int ROWS, typename O, typename S>
SXQ_DEV void pf_tile_to_lds(__amdgpu_buffer_rsrc_t src, float* dst, int wave, int lane, O&& off, S&& sw) {
    constexpr int PR = HD / 4, NI = ROWS * PR / 256;  // pieces per row, loads per wave
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int at = (wave * NI + i) * 64, r = (at + lane) / PR, p = (at + lane) % PR;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (__attribute__((address_space(3))) void*)(dst + 4 * at), 16,
                                                 off(r) + 16u * (uint32_t)(p ^ sw(r)), 0, 0, 0);
    }
}

// Zeroes rows `from` and up among the pieces this wave loaded (whose loads have completed), so
// that a probability of zero never meets an infinite value.
template <int HD, int ROWS>
SXQ_DEV void pf_zero_rows(float* dst, int wave, int lane, int from) {
    constexpr int PR = HD / 4, NI = ROWS * PR / 256;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int at = (wave * NI + i) * 64 + lane;
        if (at / PR >= from) *(float4*)(dst + 4 * at) = make_float4(0.f, 0.f, 0.f, 0.f);
    }
}

// One workgroup (256 threads) per (tile, KV group, share of the tile's rows): a tile is up to
// kPfRows / G consecutive prompt tokens of one stream (tile = {stream, first token row t0,
// count, position p0 of token t0}); its rows are r = i * G + hh (token i, query head
// g * G + hh).  Keys go through LDS 16 NP at a time, every row keeps an online softmax (running
// max m, sum l, rescaled accumulator) over blocks of 32 and masks the keys past its own position.
//
// The arithmetic is that of one multiply and one add per term, each rounded, terms in order
// (a score over the head dims, an output over the keys), whatever the split: the products
// come from v_mfma_f32_16x16x1_4b_f32 with a zero addend (four outer products of a rank-1
// update each: four head dims of 16 keys x 16 rows, or four keys of 16 dims x 16 rows), and
// the VALU adds the four blocks in order.  So the VALU issues one operation per term in
// place of two, and the matrix cores run beside it at half their rate.
//   wave w: rows 16 (w / NP) .. +15 of the workgroup's 64 / NP; keys 16 (w % NP) .. +15 of the
//   tile for the scores, which meet in LDS, and head dims HD / NP (w % NP) .. for the outputs.
//   Lane (c, b) = (lane & 15, lane >> 4) supplies element c of block b and holds row c in the
//   results.
// K is read while V loads and V while the next K loads (direct to LDS, one buffer each).
// Bound by VALU issue: 1412 ragged tokens of 32 / 8 heads of 128 in 242 us per layer (591 with
// both operations on the VALU, a score per thread and four threads per row; 104 M VALU
// instructions, 170 us of issue), 226 tokens of 14 / 2 heads of 64 in 16.4 us (66).
template <int HD, int NP>
__global__ __launch_bounds__(256, 3) void k_prefill_attn(const float* __restrict__ q, const float* __restrict__ kc,
                                                         const float* __restrict__ vc, const int4* __restrict__ tiles,
                                                         int nh, int nkv, int max_seq, int64_t kv_stream_stride,
                                                         float scale, float* __restrict__ ctx,
                                                         ActQ8_0* __restrict__ act) {
    constexpr int KT = 16 * NP, RW = 64 / NP;     // keys and rows per workgroup
    constexpr int U = HD / 4, DW = HD / NP, DT = DW / 16;  // head-dim quads; dims of a wave's outputs, in 16s
    constexpr int SS = KT + 4;  // floats per row of scores: float4-aligned, the reads hit 64 banks
    __shared__ float kt[KT * HD];  // queries first, then key tiles
    __shared__ float vt[KT * HD];
    __shared__ float st[RW * SS];
    // workgroups in the order of their tiles, which end latest first (k_prefill_tables): a tile
    // at 1024 keys takes about half of the launch, and starting one of them late left a third of
    // the CUs' time idle (310 us with each head's tiles in turn)
    constexpr int NZ = kPfRows / RW;
    const int sub = blockIdx.x % (nkv * NZ);
    const int4 tl = tiles[blockIdx.x / (nkv * NZ)];
    const int s = tl.x, t0 = tl.y, cnt = tl.z, p0 = tl.w;
    const int g = sub / NZ, G = nh / nkv, R = cnt * G, r0 = RW * (sub % NZ);
    if (r0 >= R) return;  // uniform
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, b = lane >> 4, rg = wave / NP, part = wave % NP;
    const int row = r0 + 16 * rg + c, rr = min(row, R - 1);  // rows past the tile: a copy, not stored
    const int qpos = p0 + rr / G;
    const int kend = p0 + min(r0 + RW - 1, R - 1) / G + 1;
    // reads of one element of 16 rows (keys, queries), or of DT elements of 16 lanes in 4 rows
    // (values), hit every bank
    auto ksw = [](int r) { return r & 15; };
    auto vsw = [](int r) { return DT >= 4 ? 0 : 4 * DT * (r & (4 / DT - 1)); };
    const __amdgpu_buffer_rsrc_t qrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(q + ((int64_t)t0 * nh + g * G) * HD), (short)0, (int)((uint32_t)(((cnt - 1) * nh + G) * HD) * 4u), 0x00020000);
    pf_tile_to_lds<HD, RW>(qrs, kt, wave, lane, [&](int r) {
        const int i = min(r0 + r, R - 1);
        return (uint32_t)((i / G) * nh + i % G) * (HD * 4u);
    }, ksw);
    const int64_t koff = (int64_t)s * kv_stream_stride + (int64_t)g * max_seq * HD;
    const __amdgpu_buffer_rsrc_t krs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(kc + koff), (short)0, (int)((uint32_t)kend * HD * 4u), 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(vc + koff), (short)0, (int)((uint32_t)kend * HD * 4u), 0x00020000);
    // keys past the last one load it again (their scores are masked, their values zeroed)
    auto load_k = [&](int j0) {
        pf_tile_to_lds<HD, KT>(krs, kt, wave, lane, [&](int r) { return (uint32_t)min(j0 + r, kend - 1) * (HD * 4u); }, ksw);
    };
    auto load_v = [&](int j0) {
        pf_tile_to_lds<HD, KT>(vrs, vt, wave, lane, [&](int r) { return (uint32_t)min(j0 + r, kend - 1) * (HD * 4u); }, vsw);
    };
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    float qv[U];  // head dim 4 u + b of row c
#pragma unroll
    for (int u = 0; u < U; ++u) qv[u] = kt[(16 * rg + c) * HD + 4 * (u ^ c) + b];
    lds_barrier();  // kt is free
    load_k(0);
    float m = -INFINITY, l = 0.0f;
    float o[DT][4];
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[t][e] = 0.0f;
    const float* vl = vt + b * HD + (((DW * part + DT * c) / 4) ^ vsw(b)) * 4 + (DT * c) % 4;  // key b of the tile
    for (int j0 = 0; j0 < kend; j0 += KT) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();  // the keys are here; the previous values and scores are no longer read
        load_v(j0);
        float4 sc4 = make_float4(0.f, 0.f, 0.f, 0.f);  // keys 16 part + 4 b + (0..3) of row c
        if (j0 + 16 * part < kend) {                    // uniform
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const v16f d = __builtin_amdgcn_mfma_f32_16x16x1f32(kt[(16 * part + c) * HD + 4 * (u ^ c) + b], qv[u], v16f{}, 0, 0, 0);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    sc4.x += d[4 * k];
                    sc4.y += d[4 * k + 1];
                    sc4.z += d[4 * k + 2];
                    sc4.w += d[4 * k + 3];
                }
            }
        }
        *(float4*)(st + (16 * rg + c) * SS + 16 * part + 4 * b) = sc4;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (j0 + KT > kend) pf_zero_rows<HD, KT>(vt, wave, lane, kend - j0);  // uniform: the last tile
        lds_barrier();  // the scores and values are here; the keys are no longer read
        if (j0 + KT < kend) load_k(j0 + KT);
#pragma unroll
        for (int jb = 0; jb < KT; jb += 32) {
            if (jb > 0 && j0 + jb >= kend) break;  // uniform
            float p[8], bm = -INFINITY;  // key 4 i + b of row c
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float v = st[(16 * rg + c) * SS + jb + 4 * i + b];
                p[i] = j0 + jb + 4 * i + b <= qpos ? v * scale + 0.0f : -INFINITY;
                bm = fmaxf(bm, p[i]);
            }
            float x = bm, y = bm;
            swap16(x, y);
            bm = fmaxf(x, y);
            x = y = bm;
            swap32(x, y);
            const float mn = fmaxf(m, fmaxf(x, y));
            const float corr = mn == -INFINITY ? 1.0f : expf(m - mn);
#pragma unroll
            for (int i = 0; i < 8; ++i) p[i] = p[i] == -INFINITY ? 0.0f : expf(p[i] - mn);
            // keys 8 b .. 8 b + 7 summed in order by row b of lanes, then the four sums in pairs
            float ps = 0.0f;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float a0 = p[h], a1 = p[2 + h], a2 = p[4 + h], a3 = p[6 + h];
                swap32(a0, a2);
                swap32(a1, a3);
                swap16(a0, a1);
                swap16(a2, a3);
                ps += a0;
                ps += a1;
                ps += a2;
                ps += a3;
            }
            x = y = ps;
            swap16(x, y);
            ps = x + y;
            x = y = ps;
            swap32(x, y);
            ps = x + y;
            l = l * corr + ps;
            m = mn;
#pragma unroll
            for (int t = 0; t < DT; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) o[t][e] *= corr;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                float vv[DT];
                const float* vr = vl + (jb + 4 * i) * HD;
                if constexpr (DT == 4) {
                    const float4 f = *(const float4*)vr;
                    vv[0] = f.x, vv[1] = f.y, vv[2] = f.z, vv[3] = f.w;
                } else if constexpr (DT == 2) {
                    const float2 f = *(const float2*)vr;
                    vv[0] = f.x, vv[1] = f.y;
                } else {
                    vv[0] = *vr;
                }
#pragma unroll
                for (int t = 0; t < DT; ++t) {
                    const v16f d = __builtin_amdgcn_mfma_f32_16x16x1f32(vv[t], p[i], v16f{}, 0, 0, 0);
#pragma unroll
                    for (int k = 0; k < 4; ++k)
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[t][e] += d[4 * k + e];
                }
            }
        }
    }
    // o[t][e] is head dim DW part + DT (4 b + e) + t: 4 DT consecutive dims a lane
    const int d0 = DW * part + 4 * DT * b;
    float f[4 * DT];
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) f[DT * e + t] = o[t][e] / l;
    auto head_row = [&](int r) { return (int64_t)(t0 + r / G) * nh + g * G + r % G; };  // of the context
    if (ctx && row < R) {
        float* out = ctx + head_row(rr) * HD + d0;
#pragma unroll
        for (int i = 0; i < DT; ++i) *(float4*)(out + 4 * i) = make_float4(f[4 * i], f[4 * i + 1], f[4 * i + 2], f[4 * i + 3]);
    }
    if (!act) return;  // uniform
    // the context's Q8_0 blocks for the O projection: the rows meet in kt (read last before the
    // loop's last barrier), 256 elements of them to a wave at a time
#pragma unroll
    for (int i = 0; i < DT; ++i)
        *(float4*)(kt + (16 * rg + c) * HD + d0 + 4 * i) = make_float4(f[4 * i], f[4 * i + 1], f[4 * i + 2], f[4 * i + 3]);
    lds_barrier();
#pragma unroll
    for (int i = 0; i < RW * HD / 1024; ++i) {
        const int e = 256 * (wave + 4 * i) + 4 * lane, r = r0 + e / HD;
        ActQ8_0* block = act + head_row(min(r, R - 1)) * (HD / 32) + (e % HD) / 32;
        wave_quantize_q8_0_block<false>(*(const float4*)(kt + e), lane, r < R, block);
    }
}

// One thread per token t (and per tile index): tiles in descending order of their last position;
// tokens in stream-major order, stream s's tokens at
// rows base_s .. base_s + counts[s] - 1 and positions lens[s] .. lens[s] + counts[s] - 1.
__global__ __launch_bounds__(256) void k_prefill_tables(PrefillMeta pm, int T, int2* __restrict__ tok,
                                                        int4* __restrict__ tiles, int* __restrict__ last) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    int base = 0, tbase = 0;
    for (int s = 0; s < pm.n; ++s) {
        const int c = pm.counts[s], nt = (c + pm.tile_tokens - 1) / pm.tile_tokens;
        if (t >= base && t < base + c) tok[t] = make_int2(s, pm.lens[s] + (t - base));
        if (t >= tbase && t < tbase + nt) {
            const int i0 = (t - tbase) * pm.tile_tokens, cnt = min(pm.tile_tokens, c - i0), kend = pm.lens[s] + i0 + cnt;
            // its rank: the tiles of every stream that end later, or at the same position in an
            // earlier stream (a stream's tiles end at lens + tile_tokens, lens + 2 tile_tokens, ...)
            int rank = 0;
            for (int z = 0; z < pm.n; ++z) {
                const int cz = pm.counts[z], nz = (cz + pm.tile_tokens - 1) / pm.tile_tokens;
                const int d = kend - (z < s ? 1 : 0) - pm.lens[z];  // its tiles that end at or before
                rank += nz - (d >= cz ? nz : max(d, 0) / pm.tile_tokens);
            }
            tiles[rank] = make_int4(s, base + i0, cnt, pm.lens[s] + i0);
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
                               int nkv, int hd, int max_seq, int64_t kv_stream_stride, float* ctx, void* act, hipStream_t s) {
    if (!prefill_attn_supported(nh, nkv, hd)) return hipErrorInvalidValue;
    if (n_tiles == 0) return hipSuccess;
    const float scale = (float)(1.0 / sqrt((double)hd));
    // Head dim 64: four waves per 16 rows while two of them would leave workgroups short of three
    // per CU (us at 226 tokens of 14 / 2 heads, 104 workgroups by two: 16.4 by four against
    // 23.5; 700 tokens, 312: 43.6 / 59.6; 1300 in two prompts, 580: 61 / 66; 2400 in two, 1068:
    // 179 / 165: the softmax is computed by each wave of a row).  At head dim 128 it was never
    // ahead by more than 5 % (64 KB of tiles leave two workgroups per CU).
    const bool four = hd == 64 && (int64_t)n_tiles * nkv * 2 <= 768;
#define SXQ_PF(HD, NP)                                                                                               \
    hipLaunchKernelGGL((k_prefill_attn<HD, NP>), dim3((unsigned)(n_tiles * nkv * NP)), dim3(256), 0, s, q, kc, vc,   \
                       (const int4*)tiles, nh, nkv, max_seq, kv_stream_stride, scale, ctx, (ActQ8_0*)act)
    if (hd == 128) SXQ_PF(128, 2);
    else if (four) SXQ_PF(64, 4);
    else SXQ_PF(64, 2);
#undef SXQ_PF
    return hipGetLastError();
}

hipError_t launch_gather_rows(const float* src, const int* idx, int n, int cols, float* dst, hipStream_t s) {
    hipLaunchKernelGGL(k_gather_rows, dim3(n), dim3(256), 0, s, src, idx, cols, dst);
    return hipGetLastError();
}

}  // namespace sxq
