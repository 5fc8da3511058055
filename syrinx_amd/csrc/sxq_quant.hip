// sxq_quant.hip -- block quantizers, dequantizers, weight repacking and the synthetic
// weight generator for gfx950.
//
// Bit-exactness: every float operation below is the one candle-core 0.8's CPU code
// performs (k_quants.rs from_float/to_float; utils.rs make_qkx1_quants), in the same
// order, compiled with -ffp-contract=off and IEEE division/sqrt, so results match the
// CPU byte for byte.  Call sites in the reference: QTensor::quantize at
// crates/syrinx-lm/src/cv2/load.rs:102, QTensor::dequantize at
// crates/syrinx-vocoder/src/cv2/mod.rs:172.
#include "sxq_kernels.h"
#include "sxq_quant_dev.h"

namespace sxq {

// Activation quantization kernel: rows x [m, k] (row stride ldx floats) -> blocks.
// One wave per 256-element chunk.  out_canon: canonical Candle blocks [m][k/bs];
// otherwise the device layout ActQ8K/ActQ8_0 [m][k/bs].
// XT: float, or uint16_t for bf16 rows.  V: rows are aligned for the four-element load.
template <bool V, typename XT>
SXQ_DEV float4 act_load4(const XT* p) {
    if constexpr (sizeof(XT) == 4) {
        return *(const float4*)p;
    } else {
        ushort4 u;
        if (V) u = *(const ushort4*)p;
        else u = make_ushort4(p[0], p[1], p[2], p[3]);
        return make_float4(__uint_as_float((uint32_t)u.x << 16), __uint_as_float((uint32_t)u.y << 16),
                           __uint_as_float((uint32_t)u.z << 16), __uint_as_float((uint32_t)u.w << 16));
    }
}
template <int VDT, bool CANON, typename XT = float, bool V = true>
__global__ __launch_bounds__(256) void k_quantize_act(const XT* __restrict__ x, int64_t ldx, int m,
                                                      int k, void* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const int chunk = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int chunks_per_row = (k + 255) / 256;
    const int row = blockIdx.y;
    if (row >= m || chunk >= chunks_per_row) return;
    const int e0 = chunk * 256 + 4 * lane;
    const XT* xr = x + (int64_t)row * ldx;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (e0 < k) v = act_load4<V>(xr + e0);  // k is a multiple of 32, so 4 | k
    if (VDT == kQ8K) {
        const int nb = k / 256;
        char* base = (char*)out + ((int64_t)row * nb + chunk) * (CANON ? sizeof(BlockQ8K) : sizeof(ActQ8K));
        wave_quantize_q8k<CANON>(v, lane, base);
    } else {
        const int nb = k / 32;
        const int blk0 = chunk * 8;
        char* base = (char*)out + ((int64_t)row * nb + blk0) * (CANON ? sizeof(BlockQ8_0) : sizeof(ActQ8_0));
        wave_quantize_q8_0<CANON>(v, lane, blk0 + (lane >> 3) < nb, base);
    }
}

hipError_t launch_quantize_act(int vdt, bool canon, const float* x, int64_t ldx, int m, int k, void* out,
                               hipStream_t s) {
    const int chunks = (k + 255) / 256;
    dim3 grid((chunks + 3) / 4, m);
    if (vdt == kQ8K) {
        if (canon) hipLaunchKernelGGL((k_quantize_act<kQ8K, true>), grid, dim3(256), 0, s, x, ldx, m, k, out);
        else hipLaunchKernelGGL((k_quantize_act<kQ8K, false>), grid, dim3(256), 0, s, x, ldx, m, k, out);
    } else {
        if (canon) hipLaunchKernelGGL((k_quantize_act<kQ8_0, true>), grid, dim3(256), 0, s, x, ldx, m, k, out);
        else hipLaunchKernelGGL((k_quantize_act<kQ8_0, false>), grid, dim3(256), 0, s, x, ldx, m, k, out);
    }
    return hipGetLastError();
}

hipError_t launch_quantize_act_bf16(int vdt, const uint16_t* x, int64_t ldx, int m, int k, void* out, hipStream_t s) {
    const dim3 grid(((k + 255) / 256 + 3) / 4, m);
    const bool vec = ((uintptr_t)x & 7) == 0 && ldx % 4 == 0;
#define SXQ_QUANT_BF16(VDT, V) \
    hipLaunchKernelGGL((k_quantize_act<VDT, false, uint16_t, V>), grid, dim3(256), 0, s, x, ldx, m, k, out)
    if (vdt == kQ8K) {
        if (vec) SXQ_QUANT_BF16(kQ8K, true);
        else SXQ_QUANT_BF16(kQ8K, false);
    } else {
        if (vec) SXQ_QUANT_BF16(kQ8_0, true);
        else SXQ_QUANT_BF16(kQ8_0, false);
    }
#undef SXQ_QUANT_BF16
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// Weight from_float (QTensor::quantize on the device), canonical output.
//
// Q8_0 and Q4_0: eight lanes per block, four elements each, so a wave reads 1 KB and writes
// 272 / 144 bytes contiguously.  Memory-bound: a 2560 x 9728 matrix in 24.1 / 23.9 us (5.2 /
// 4.8 TB/s), against 39.4 / 30.7 us with one thread per block reading 128 B strides and
// writing single bytes.  V: x is 16-byte aligned and `out` 2-byte aligned (any tensor's own
// storage); otherwise element loads and byte stores.
template <bool V>
SXQ_DEV float4 load4(const float* p) {
    if (V) return *(const float4*)p;
    return make_float4(p[0], p[1], p[2], p[3]);
}
// n bytes of w (little-endian dwords) to o: 2-byte stores, or single bytes.
template <bool V>
SXQ_DEV void store_dword(uint8_t* o, uint32_t w) {
    if (V) {
        *(uint16_t*)o = (uint16_t)w;
        *(uint16_t*)(o + 2) = (uint16_t)(w >> 16);
    } else {
        for (int i = 0; i < 4; ++i) o[i] = (uint8_t)(w >> (8 * i));
    }
}
template <bool V>
SXQ_DEV void store_half(uint8_t* o, uint32_t w) {
    if (V) {
        *(uint16_t*)o = (uint16_t)w;
    } else {
        o[0] = (uint8_t)w;
        o[1] = (uint8_t)(w >> 8);
    }
}

template <bool V>
__global__ __launch_bounds__(256) void k_from_float_q8_0(const float* __restrict__ x, int64_t nblocks,
                                                         uint8_t* __restrict__ out) {
    const int64_t b = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 3;
    const int l = threadIdx.x & 7;
    if (b >= nblocks) return;  // a block's eight lanes leave together
    const float4 v = load4<V>(x + b * 32 + 4 * l);
    // fmaxf ignores NaN, so the order of the maxima does not matter
    float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    amax = fmaxf(amax, 0.0f);
    for (int o = 1; o < 8; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
    const float d = amax / 127.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    const uint32_t w = (uint32_t)(uint8_t)sat_i8(roundf(v.x * id)) | (uint32_t)(uint8_t)sat_i8(roundf(v.y * id)) << 8 |
                       (uint32_t)(uint8_t)sat_i8(roundf(v.z * id)) << 16 | (uint32_t)(uint8_t)sat_i8(roundf(v.w * id)) << 24;
    uint8_t* o = out + b * 34;
    if (l == 0) store_half<V>(o, f32_to_f16_bits(d));
    store_dword<V>(o + 2 + 4 * l, w);
}

template <bool V>
__global__ __launch_bounds__(256) void k_from_float_q4_0(const float* __restrict__ x, int64_t nblocks,
                                                         uint8_t* __restrict__ out) {
    const int64_t b = ((int64_t)blockIdx.x * 256 + threadIdx.x) >> 3;
    const int l = threadIdx.x & 7;
    if (b >= nblocks) return;
    const float4 v4 = load4<V>(x + b * 32 + 4 * l);
    const float v[4] = {v4.x, v4.y, v4.z, v4.w};
    // the first element of the largest magnitude (a NaN never compares larger)
    float amax = 0.0f, mx = 0.0f;
    int at = 4 * l;
    for (int i = 0; i < 4; ++i) {
        const float a = fabsf(v[i]);
        if (amax < a) { amax = a; mx = v[i]; at = 4 * l + i; }
    }
    for (int o = 1; o < 8; o <<= 1) {
        const float a2 = __shfl_xor(amax, o, 64), m2 = __shfl_xor(mx, o, 64);
        const int at2 = __shfl_xor(at, o, 64);
        if (amax < a2 || (amax == a2 && at2 < at)) { amax = a2; mx = m2; at = at2; }
    }
    const float d = mx / -8.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    uint32_t q = 0;
    for (int i = 0; i < 4; ++i) {
        // Rust `(x + 8.5) as u8`: truncate toward zero, saturating at 0 and 255 (NaN -> 0).
        const float t = v[i] * id + 8.5f;
        const int a = t != t ? 0 : (t <= 0.0f ? 0 : (t >= 255.0f ? 255 : (int)t));
        q |= (uint32_t)(a > 15 ? 15 : a) << (8 * i);
    }
    const uint32_t hi = __shfl_xor(q, 4, 64);  // byte j holds elements j and j + 16
    uint8_t* o = out + b * 18;
    if (l == 0) store_half<V>(o, f32_to_f16_bits(d));
    if (l < 4) store_dword<V>(o + 2 + 4 * l, q | (hi << 4));
}

// make_qkx1_quants(15, 5, x[32]) for one Q4_K sub-block (utils.rs): one thread runs the
// sequential algorithm so every float sum has Candle's order.
SXQ_DEV int nearest_int(float v) {
    const float r = roundf(v);
    return r != r ? 0 : (r >= 2147483647.0f ? 2147483647 : (r <= -2147483648.0f ? (int)0x80000000u : (int)r));
}
// nearest_int(v) clamped to 0..15, as a float: half-away rounding only matters above zero, where
// it is trunc(v + the float below 0.5) (checked for every f32); a NaN gives 0 and an infinity
// its bound, as the clamped int does.
SXQ_DEV float level15(float v) { return __builtin_amdgcn_fmed3f(truncf(v + 0x1.fffffep-2f), 0.0f, 15.0f); }
// level15(a / d), y = RN(1 / d): with a faithful q0 = a y the quotient rounded once is
// q0 + (a - q0 d) y (Markstein); a q0 too large for that (or not finite) is at a bound anyway.
SXQ_DEV float level15_div(float a, float d, float y) {
    const float q0 = a * y;
    const float q = __builtin_fmaf(__builtin_fmaf(-d, q0, a), y, q0);
    return level15(fabsf(q0) < 32.0f ? q : q0);
}
// f32 bits <-> the integer of the same total order (its own inverse)
SXQ_DEV int total_key(int a) { return a ^ (int)(((unsigned)(a >> 31)) >> 1); }
SXQ_DEV void make_qkx1_quants(const float (&x)[32], float* scale_out, float* min_out) {
    int kmin = total_key(__builtin_bit_cast(int, x[0])), kmax = kmin;
#pragma unroll
    for (int i = 1; i < 32; ++i) {
        const int k = total_key(__builtin_bit_cast(int, x[i]));
        kmin = k < kmin ? k : kmin;
        kmax = k > kmax ? k : kmax;
    }
    const float mn = __builtin_bit_cast(float, total_key(kmin)), mx = __builtin_bit_cast(float, total_key(kmax));
    *scale_out = 0.0f;
    *min_out = 0.0f;
    if (mx == mn) return;
    float L[32];  // levels, whole numbers 0..15
#pragma unroll
    for (int i = 0; i < 32; ++i) L[i] = 0.0f;
    float min = fminf(mn, 0.0f);
    float iscale = 15.0f / (mx - min);
    float scale = 0.0f;
    for (int it = 0; it < 5; ++it) {
        float sumlx = 0.0f, suml2 = 0.0f;  // suml2: at most 32 * 225, exact either way
        bool changed = false;
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            const float dx = x[i] - min;
            const float li = level15(iscale * dx);
            changed = changed || li != L[i];
            L[i] = li;
            sumlx += dx * li;
            suml2 = __builtin_fmaf(li, li, suml2);
        }
        scale = sumlx / suml2;
        float sum = -0.0f;
#pragma unroll
        for (int i = 0; i < 32; ++i) sum += x[i] - scale * L[i];
        min = sum / 32.0f;
        if (min > 0.0f) min = 0.0f;
        iscale = 1.0f / scale;
        if (!changed) break;
    }
    *scale_out = scale;
    *min_out = -min;
}

SXQ_DEV void get_scale_min_k4(int j, const uint8_t* q, int& d, int& m) {
    if (j < 4) {
        d = q[j] & 63;
        m = q[j + 4] & 63;
    } else {
        d = (q[j + 4] & 0xF) | ((q[j - 4] >> 6) << 4);
        m = (q[j + 4] >> 4) | ((q[j] >> 6) << 4);
    }
}

// One thread per 32-element sub-block, its values and levels in registers; the eight lanes
// of a super-block share the scale search's results by shuffles and each packs its own
// nibbles.  The search is a serial chain of float sums per sub-block (up to 5 x 64 adds in
// Candle's order), so the parallelism is over sub-blocks: VALU-bound.  With a workgroup per
// super-block (eight of its 256 threads searching) a 2560 x 9728 matrix took 9666 us; this runs
// it in 49 us (56 with the rounding and the final divisions spelled out: 16 VALU operations per
// element and round where there are 12 now).  V: x and out are 16-byte aligned; otherwise
// element loads and byte stores.
template <bool V>
__global__ __launch_bounds__(256) void k_from_float_q4k(const float* __restrict__ x, int64_t nblocks,
                                                        uint8_t* __restrict__ out) {
    const int64_t sub = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t b = sub >> 3;
    const int j = threadIdx.x & 7;
    if (b >= nblocks) return;  // a super-block's eight lanes leave together
    float xs[32];
#pragma unroll
    for (int i = 0; i < 32; i += 4) {
        const float4 v = load4<V>(x + sub * 32 + i);
        xs[i] = v.x;
        xs[i + 1] = v.y;
        xs[i + 2] = v.z;
        xs[i + 3] = v.w;
    }
    float scale, min;
    make_qkx1_quants(xs, &scale, &min);
    float max_scale = fmaxf(scale, 0.0f), max_min = fmaxf(min, 0.0f);  // fmaxf ignores NaN
    for (int o = 1; o < 8; o <<= 1) {
        max_scale = fmaxf(max_scale, __shfl_xor(max_scale, o, 64));
        max_min = fmaxf(max_min, __shfl_xor(max_min, o, 64));
    }
    const float inv_scale = max_scale > 0.0f ? 63.0f / max_scale : 0.0f;
    const float inv_min = max_min > 0.0f ? 63.0f / max_min : 0.0f;
    const int lsi = nearest_int(inv_scale * scale), lmi = nearest_int(inv_min * min);
    const uint32_t ls = (uint8_t)(lsi < 63 ? lsi : 63), lm = (uint8_t)(lmi < 63 ? lmi : 63);
    // header bytes: lane j < 4 holds scales[j], [j + 4] and [j + 8]; lane j + 4 the same copies
    const uint32_t ls4 = __shfl_xor(ls, 4, 64), lm4 = __shfl_xor(lm, 4, 64);
    const bool up = j >= 4;
    const uint32_t ls_lo = up ? ls4 : ls, ls_hi = up ? ls : ls4, lm_lo = up ? lm4 : lm, lm_hi = up ? lm : lm4;
    const uint32_t b0 = (ls_lo | ((ls_hi >> 4) << 6)) & 0xFFu, b1 = (lm_lo | ((lm_hi >> 4) << 6)) & 0xFFu;
    const uint32_t b2 = (ls_hi & 0xFu) | ((lm_hi & 0xFu) << 4);
    const uint32_t sc = up ? (b2 & 0xFu) | ((b0 >> 6) << 4) : b0 & 63u;
    const uint32_t m = up ? (b2 >> 4) | ((b1 >> 6) << 4) : b1 & 63u;
    const uint16_t dh = f32_to_f16_bits(max_scale / 63.0f), mh = f32_to_f16_bits(max_min / 63.0f);
    const float d = f16_bits_to_f32(dh) * (float)sc;
    const float dm = f16_bits_to_f32(mh) * (float)m;
    const float y = 1.0f / d;
    uint32_t w[8];  // this sub-block's levels, a byte each
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        w[i] = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (d != 0.0f) w[i] |= (uint32_t)level15_div(xs[4 * i + t] + dm, d, y) << (8 * t);
    }
    // byte l of 64-element chunk c: sub-block 2c's level l below, 2c + 1's above; the lower
    // lane of a pair stores the first 16 bytes of the chunk, the upper one the rest
    uint32_t qs[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t lo = __shfl_xor(w[i], 1, 64), hi = __shfl_xor(w[4 + i], 1, 64);
        qs[i] = (j & 1) ? (hi | (w[4 + i] << 4)) : (w[i] | (lo << 4));
    }
    uint32_t h0 = b0 << (8 * (j & 3)), h1 = b1 << (8 * (j & 3)), h2 = b2 << (8 * (j & 3));
    for (int o = 1; o < 4; o <<= 1) {
        h0 |= __shfl_xor(h0, o, 64);
        h1 |= __shfl_xor(h1, o, 64);
        h2 |= __shfl_xor(h2, o, 64);
    }
    const uint4 hdr = make_uint4((uint32_t)dh | ((uint32_t)mh << 16), h0, h1, h2);
    uint8_t* o = out + b * 144;
    if (V) {
        if (j == 0) *(uint4*)o = hdr;
        *(uint4*)(o + 16 + 16 * j) = make_uint4(qs[0], qs[1], qs[2], qs[3]);
    } else {
        const uint32_t hw[4] = {hdr.x, hdr.y, hdr.z, hdr.w};
        for (int i = 0; i < 16; ++i) {
            if (j == 0) o[i] = (uint8_t)(hw[i >> 2] >> (8 * (i & 3)));
            o[16 + 16 * j + i] = (uint8_t)(qs[i >> 2] >> (8 * (i & 3)));
        }
    }
}

hipError_t launch_from_float(int dt, const float* x, int64_t nblocks, void* out, hipStream_t s) {
    if (nblocks <= 0) return hipSuccess;
    const bool vec = ((uintptr_t)x & 15) == 0 && ((uintptr_t)out & (dt == kQ4K ? 15 : 1)) == 0;
    const dim3 grid((unsigned)((nblocks + 31) / 32));  // eight lanes per block (or super-block)
#define SXQ_FROM_FLOAT(K)                                                                                   \
    do {                                                                                                    \
        if (vec) hipLaunchKernelGGL((K<true>), grid, dim3(256), 0, s, x, nblocks, (uint8_t*)out);           \
        else hipLaunchKernelGGL((K<false>), grid, dim3(256), 0, s, x, nblocks, (uint8_t*)out);              \
    } while (0)
    if (dt == kQ8_0) SXQ_FROM_FLOAT(k_from_float_q8_0);
    else if (dt == kQ4_0) SXQ_FROM_FLOAT(k_from_float_q4_0);
    else if (dt == kQ4K) SXQ_FROM_FLOAT(k_from_float_q4k);
    else if (dt == kQ8K) {
        // Q8_K is an activation type; rows of 256 are quantized one wave each.
        return launch_quantize_act(kQ8K, true, x, 256, (int)nblocks, 256, out, s);
    } else return hipErrorInvalidValue;
#undef SXQ_FROM_FLOAT
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// to_float from canonical blocks.  One thread per element.
__global__ void k_to_float(int dt, const uint8_t* __restrict__ blocks, int64_t nelem, float* __restrict__ y) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nelem) return;
    if (dt == kQ8_0) {
        const uint8_t* b = blocks + (e / 32) * 34;
        const float d = f16_bits_to_f32((uint16_t)(b[0] | (b[1] << 8)));
        y[e] = (float)(int8_t)b[2 + (e % 32)] * d;
    } else if (dt == kQ4_0) {
        const uint8_t* b = blocks + (e / 32) * 18;
        const float d = f16_bits_to_f32((uint16_t)(b[0] | (b[1] << 8)));
        const int i = (int)(e % 32);
        const int q = i < 16 ? (b[2 + i] & 0xF) : (b[2 + i - 16] >> 4);
        y[e] = (float)(q - 8) * d;
    } else if (dt == kQ8K) {
        const uint8_t* b = blocks + (e / 256) * 292;
        const float d = __builtin_bit_cast(float, (uint32_t)(b[0] | (b[1] << 8) | (b[2] << 16) | ((uint32_t)b[3] << 24)));
        y[e] = d * (float)(int8_t)b[4 + (e % 256)];
    } else if (dt == kQ4K) {
        const uint8_t* b = blocks + (e / 256) * 144;
        const int i = (int)(e % 256);
        const int c = i / 64, p = i % 64, hi = p >= 32, l = p & 31;
        const float d = f16_bits_to_f32((uint16_t)(b[0] | (b[1] << 8)));
        const float dmin = f16_bits_to_f32((uint16_t)(b[2] | (b[3] << 8)));
        int sc, m;
        get_scale_min_k4(2 * c + hi, b + 4, sc, m);
        const float d1 = d * (float)sc, m1 = dmin * (float)m;
        const uint8_t qb = b[16 + 32 * c + l];
        const int q = hi ? (qb >> 4) : (qb & 0xF);
        y[e] = d1 * (float)q - m1;
    }
}

hipError_t launch_to_float(int dt, const void* blocks, int64_t nelem, float* y, hipStream_t s) {
    if (nelem <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_to_float, dim3((nelem + 255) / 256), dim3(256), 0, s, dt, (const uint8_t*)blocks, nelem, y);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// Repack canonical weight blocks into the device layout (and back).  One thread per block.
__global__ void k_repack(int dt, const uint8_t* __restrict__ canon, int64_t nblocks, uint8_t* __restrict__ hdr,
                         uint8_t* __restrict__ qs, bool to_device) {
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nblocks) return;
    if (dt == kQ4K) {
        uint8_t* cb = (uint8_t*)canon + b * 144;
        uint8_t* h = hdr + b * 16;
        uint8_t* q = qs + b * 128;
        if (to_device) {
            for (int i = 0; i < 16; ++i) h[i] = cb[i];
            // device byte (4*(4l + c) + t) <- canonical qs byte 32c + l + 8t
            for (int l = 0; l < 8; ++l)
                for (int c = 0; c < 4; ++c)
                    for (int t = 0; t < 4; ++t) q[4 * (4 * l + c) + t] = cb[16 + 32 * c + l + 8 * t];
        } else {
            for (int i = 0; i < 16; ++i) cb[i] = h[i];
            for (int l = 0; l < 8; ++l)
                for (int c = 0; c < 4; ++c)
                    for (int t = 0; t < 4; ++t) cb[16 + 32 * c + l + 8 * t] = q[4 * (4 * l + c) + t];
        }
    } else {
        const int qb = dt == kQ8_0 ? 32 : 16, tb = qb + 2;
        uint8_t* cb = (uint8_t*)canon + b * tb;
        if (to_device) {
            hdr[2 * b] = cb[0];
            hdr[2 * b + 1] = cb[1];
            for (int i = 0; i < qb; ++i) qs[b * qb + i] = cb[2 + i];
        } else {
            cb[0] = hdr[2 * b];
            cb[1] = hdr[2 * b + 1];
            for (int i = 0; i < qb; ++i) cb[2 + i] = qs[b * qb + i];
        }
    }
}

hipError_t launch_repack(int dt, const void* canon, int64_t nblocks, void* hdr, void* qs, bool to_device, hipStream_t s) {
    if (nblocks <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_repack, dim3((nblocks + 255) / 256), dim3(256), 0, s, dt, (const uint8_t*)canon, nblocks,
                       (uint8_t*)hdr, (uint8_t*)qs, to_device);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// Synthetic weights: element i of stream `seed` is N(mean, std) from a counter-based
// SplitMix64 pair and the Box-Muller transform (f64), rounded to f32.
SXQ_DEV uint64_t splitmix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
__global__ void k_fill_normal(float* __restrict__ y, int64_t n, uint64_t seed, float mean, float stdv) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint64_t base = seed * 0xD1B54A32D192ED03ull;
    const uint64_t a = splitmix64(base + 2 * (uint64_t)i), b = splitmix64(base + 2 * (uint64_t)i + 1);
    const double u1 = ((double)(a >> 11) + 1.0) * 0x1.0p-53;
    const double u2 = (double)(b >> 11) * 0x1.0p-53;
    const double z = sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
    y[i] = (float)((double)mean + (double)stdv * z);
}

__global__ void k_bf16_to_f32(const uint16_t* __restrict__ x, int64_t n, float* __restrict__ y) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = __uint_as_float((uint32_t)x[i] << 16);
}

hipError_t launch_bf16_to_f32(const uint16_t* x, int64_t n, float* y, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_bf16_to_f32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, n, y);
    return hipGetLastError();
}

hipError_t launch_fill_normal(float* y, int64_t n, uint64_t seed, float mean, float stdv, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_normal, dim3((n + 255) / 256), dim3(256), 0, s, y, n, seed, mean, stdv);
    return hipGetLastError();
}

}  // namespace sxq
