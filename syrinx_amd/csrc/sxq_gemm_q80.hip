// sxq_gemm_q80.hip -- QMatMul over Q8_0 / Q4_0 weights for five rows and more, on the int8
// matrix cores, bit-identical to Candle's vec-dot.
//
// A prompt's projections and the steps of several streams (QMatMul::forward with M > 4 rows;
// the reference calls it at crates/syrinx-lm/src/cv2/mod.rs:197, whose weights load as Q4_0 at
// crates/syrinx-lm/src/cv2/load.rs:101-104) are a GEMM.  Candle computes every output as
// sum over blocks b of ((f32)S_b * d_w) * d_a, where S_b is the integer dot of one
// 32-element block of the weight row (int8 Q8_0 quants, or Q4_0 nibbles minus 8) with the
// Q8_0-quantized activation row, added block after block in f32.  One int8 MFMA of K depth
// 32 is exactly that integer dot for a tile of (row, weight row) pairs over one block:
// integer sums are exact in any order.  The two multiplies and the add of each block then
// run in Candle's order, so the outputs are Candle's bits at every row count, unlike an f16
// GEMM (which rounds both operands).  The float fold is 4 VALU instructions per output per
// block against 1/16 of an MFMA, so with enough tiles the work is bound by VALU issue.
//
// The adds of one output are a serial chain over its blocks, and three kernels split the rest:
//  * k_gemm_q80: one wave per 32 x 32 tile, the chain in its registers; ~0.27 us per block
//    where a SIMD holds one wave, so this is for shapes with many tiles.
//  * k_gemm_q80_mid: one wave per 16 x 16 tile, likewise: four times the waves.
//  * k_gemm_q80_split: the eight waves of a workgroup take different blocks of one 16 x 16
//    tile, leave the products in LDS and one thread per output adds them in block order.
//    Eight times the parallelism per tile at about twice the work per output: for few tiles.
// One kernel (64 x 128 tiles, operands one block ahead in registers, 1.1 us per block) for 128
// rows and more and the GEMV four rows per launch below took: 896 x 4864 at 8 / 50 / 226 rows
// 12.9 / 69 / 166 us (now 10.8 / 11.4 / 21.3), 9728 x 896 12.5 / 63 / 45 (7.6 / 10.4 / 20.6), 2048 x
// 1024 Q4_0 at 500 rows 46.7 (14.7), all with the activation quantizer's launch.
#include "sxq_kernels.h"
#include "sxq_q80_stage.h"
#include "sxq_quant_dev.h"

namespace sxq {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// Q4_0 nibbles (one per byte, 0..15) as int8 q - 8: (q + 0x78) ^ 0x80 per byte (the add never
// carries into the next byte).
SXQ_DEV uint32_t nib_i8(uint32_t q) { return ((q & 0x0F0F0F0Fu) + 0x78787878u) ^ 0x80808080u; }

// An f16 block scale as f32, exact: one conversion (f16_bits_to_f32 takes branches).
SXQ_DEV float f16_scale(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }

// Workgroups are numbered so that every row tile of one weight tile lands on the same XCD
// (workgroup id mod 8), whose L2 then serves the weight tile's re-reads.
SXQ_DEV void xcd_tile(int id, int tiles_m, int& mt, int& nt) {
    const int slot = id >> 3;
    nt = (slot / tiles_m) * 8 + (id & 7);
    mt = slot % tiles_m;
}

// ---- few rows or long K: blocks over the waves, chains in LDS ---------------------------

constexpr int kSpN = 16;           // weight rows per workgroup
constexpr int kSpWaves = 8;        // 512 threads
constexpr int kSpRow = 20;         // floats per weight row of a block's products (16 rows + padding:
                                   // 80 B keeps the float4 writes and the column reads conflict-free)
constexpr int kSpTile = kSpN * kSpRow;

// A chunk is JB consecutive blocks for each wave.  A chunk's weights (1 KB contiguous per
// Q8_0 row at JB = 4), scales and activation blocks come by coalesced loads, one or two
// chunks ahead, into registers and then LDS (rows padded by 16 B: the lanes' operand reads hit every bank
// once).  Loading the operands straight into their lanes instead (16 rows' lines touched per
// instruction) ran 896 x 4864 at 8 rows in 22.6 us against 12.1.  Lane (r, g) = (lane & 15,
// lane >> 4) feeds v_mfma_i32_16x16x32_i8 with weight row n0 + r and activation row m0 + r,
// eight elements of the block each (Q8_0: elements 8g .. 8g+7; Q4_0: the nibbles of bytes 4g
// .. 4g+3, elements 4g .. 4g+3 and 16 + 4g .. 16 + 4g+3), and gets the integer dots of weight
// row r with rows 4g .. 4g+3.  The barriers wait for LDS only: loads stay in flight.  Loads
// are of clamped rows and blocks; what those give is never added or stored.
template <bool Q4, int JB>
struct SplitShape {
    static constexpr int KC = JB * kSpWaves;                // blocks per chunk
    static constexpr int WB = Q4 ? 16 : 32;                 // quant bytes per weight block
    static constexpr int WROW = KC * WB + 16;               // LDS bytes of a weight row
    static constexpr int AROW = KC * (int)sizeof(ActQ8_0) + 16;
    static constexpr int WP = kSpN * KC * WB / 16;          // 16-byte pieces of a chunk: weights
    static constexpr int AP = 16 * KC * 3;                  // activations
    static constexpr int THREADS = 64 * kSpWaves;
    static constexpr size_t lds = (size_t)kSpN * WROW + (size_t)16 * AROW + (size_t)kSpN * (KC + 1) * 4 +
                                  (size_t)KC * kSpTile * 4;
};

template <bool Q4, int JB>
__global__ __launch_bounds__(64 * kSpWaves) void k_gemm_q80_split(const ActQ8_0* __restrict__ act, int M, int nb,
                                                                  const uint16_t* __restrict__ wd,
                                                                  const uint8_t* __restrict__ wqs, int N, int tiles_m,
                                                                  int tiles_n, float* y, int64_t ldy,
                                                                  const float* __restrict__ bias, const float* res,
                                                                  int64_t ldr) {
    using S = SplitShape<Q4, JB>;
    constexpr int KC = S::KC, T = S::THREADS, AHEAD = JB == 4 ? 2 : 1;
    constexpr int NW = (S::WP + T - 1) / T, NA = (S::AP + T - 1) / T, ND = (kSpN * KC + T - 1) / T;
    extern __shared__ __align__(16) char smem[];
    char* sw = smem;                                        // [16][WROW]
    char* sa = sw + kSpN * S::WROW;                         // [16][AROW], ActQ8_0 blocks
    float* pr = (float*)(sa + 16 * S::AROW);           // [KC][16][kSpRow] products
    float* sd = pr + KC * kSpTile;                     // [16][KC + 1] weight scales
    int mt, nt;
    xcd_tile(blockIdx.x, tiles_m, mt, nt);
    if (nt >= tiles_n) return;  // uniform: padding of the weight tiles to a multiple of 8
    const int m0 = mt * 16, n0 = nt * kSpN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 15, g = lane >> 4;

    struct Regs {
        v4i w[NW], a[NA];
        uint16_t d[ND];
    };
    auto stage_load = [&](Regs& k, int c0) {
#pragma unroll
        for (int i = 0; i < NW; ++i) {  // piece u: row u / (pieces per row), in block order
            constexpr int P = KC * S::WB / 16, PB = S::WB / 16;
            const int u = min(tid + T * i, S::WP - 1), row = u / P, p = u % P;
            const int64_t b = (int64_t)min(n0 + row, N - 1) * nb + min(c0 + p / PB, nb - 1);
            k.w[i] = *(const v4i*)(wqs + b * S::WB + 16 * (p % PB));
        }
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            const int u = min(tid + T * i, kSpN * KC - 1);
            k.d[i] = wd[(int64_t)min(n0 + u / KC, N - 1) * nb + min(c0 + u % KC, nb - 1)];
        }
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int u = min(tid + T * i, S::AP - 1), row = u / (3 * KC), p = u % (3 * KC);
            const ActQ8_0* ab = act + (int64_t)min(m0 + row, M - 1) * nb + min(c0 + p / 3, nb - 1);
            k.a[i] = *((const v4i*)ab + p % 3);
        }
    };
    auto stage_store = [&](const Regs& k) {
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            constexpr int P = KC * S::WB / 16;
            const int u = min(tid + T * i, S::WP - 1);
            *(v4i*)(sw + (u / P) * S::WROW + 16 * (u % P)) = k.w[i];
        }
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            const int u = min(tid + T * i, kSpN * KC - 1);
            sd[(u / KC) * (KC + 1) + u % KC] = f16_scale(k.d[i]);
        }
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int u = min(tid + T * i, S::AP - 1);
            *(v4i*)(sa + (u / (3 * KC)) * S::AROW + 16 * (u % (3 * KC))) = k.a[i];
        }
    };
    auto products = [&]() {
        const v4i zero = {};
#pragma unroll
        for (int j = 0; j < JB; ++j) {
            const int b = JB * wave + j;
            uint32_t w0, w1;
            if (Q4) {
                const uint32_t q = *(const uint32_t*)(sw + r * S::WROW + b * 16 + 4 * g);
                w0 = nib_i8(q);
                w1 = nib_i8(q >> 4);
            } else {
                const uint2 v = *(const uint2*)(sw + r * S::WROW + b * 32 + 8 * g);
                w0 = v.x;
                w1 = v.y;
            }
            const long wv = (long)((uint64_t)w0 | ((uint64_t)w1 << 32));
            const float dw = sd[r * (KC + 1) + b];
            const char* ab = sa + r * S::AROW + b * (int)sizeof(ActQ8_0);
            uint32_t a0, a1;
            if (Q4) {
                a0 = *(const uint32_t*)(ab + 4 * g);
                a1 = *(const uint32_t*)(ab + 16 + 4 * g);
            } else {
                const uint2 v = *(const uint2*)(ab + 8 * g);
                a0 = v.x;
                a1 = v.y;
            }
            const long av = (long)((uint64_t)a0 | ((uint64_t)a1 << 32));
            const v4i s = __builtin_amdgcn_mfma_i32_16x16x32_i8(av, wv, zero, 0, 0, 0);
            const char* db = sa + 4 * g * S::AROW + b * (int)sizeof(ActQ8_0) + 32;  // rows 4g .. 4g + 3: their d
            float p[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] = ((float)s[i] * dw) * *(const float*)(db + i * S::AROW);
            *(float4*)(pr + b * kSpTile + r * kSpRow + 4 * g) = make_float4(p[0], p[1], p[2], p[3]);
        }
    };

    // one output per thread of the first four waves: row om, weight row on
    const int om = (tid & 255) >> 4, on = tid & 15;
    const float* pc = pr + on * kSpRow + om;
    const bool fold = tid < 256;
    float acc = 0.0f;
    auto chunk = [&](Regs& k, int c0) {
        stage_store(k);  // the previous chunk's operand reads are behind its second barrier
        lds_barrier();
        if (c0 + AHEAD * KC < nb) stage_load(k, c0 + AHEAD * KC);  // uniform
        products();
        lds_barrier();
        if (fold) {
            const int kc = nb - c0;
            if (kc >= KC) {
#pragma unroll
                for (int b = 0; b < KC; ++b) acc = acc + pc[b * kSpTile];
            } else {
#pragma unroll 4
                for (int b = 0; b < kc; ++b) acc = acc + pc[b * kSpTile];
            }
        }
    };
    // Where a workgroup has its CU to itself (JB = 4) the loads go two chunks ahead: a chunk takes
    // less time than they do (896 x 4864 at 8 rows 11.5 -> 10.9 us).  With three workgroups per
    // CU the others cover them (2560 x 9728 at 32 rows 26.9 us, 29.0 with two sets of registers).
    Regs k0;
    stage_load(k0, 0);
    if constexpr (AHEAD == 2) {
        Regs k1;
        if (KC < nb) stage_load(k1, KC);
        for (int c0 = 0; c0 < nb; c0 += 2 * KC) {
            chunk(k0, c0);
            if (c0 + KC >= nb) break;  // uniform
            chunk(k1, c0 + KC);
        }
    } else {
        for (int c0 = 0; c0 < nb; c0 += KC) chunk(k0, c0);
    }
    const int m = m0 + om, n = n0 + on;
    if (fold && m < M && n < N) {
        float v = bias ? acc + bias[n] : acc;
        if (res) v = res[(int64_t)m * ldr + n] + v;
        y[(int64_t)m * ldy + n] = v;
    }
}

// ---- many tiles: one wave per 32 x 32 tile -----------------------------------------

constexpr int kQBM = 64;  // activation rows, and weight rows, per workgroup tile
constexpr int kQKC = 4;   // blocks per LDS stage

// y[m][n] = sum_b ((f32)S_b[m][n] * d_w[n][b]) * d_a[m][b] (+ bias[n], then res[m][n] + that).
// act: the Q8_0 activation blocks [M][nb] (ActQ8_0: quants, f32 d).  Weight device layout:
// wd[n * nb + b] f16 scales, wqs the quants (32 B per Q8_0 block, 16 B per Q4_0 block).
// One workgroup of 256 threads per 64 x 64 tile; wave w covers rows 32 (w & 1) .. +31 and
// weight rows 32 (w >> 1) .. +31 with v_mfma_i32_32x32x32_i8: lane (l, h)
// feeds A row l and B weight row l, elements 16h .. 16h+15 of the block; result i is row
// 8 (i / 4) + 4 h + i % 4, weight row l.  Four blocks at a time go through LDS (double
// buffered, one barrier per stage; the next stage's loads are in flight while a stage is
// computed): 16-byte pieces, piece p of row r stored at p ^ ((r >> 1) & 7), which spreads any
// 16 consecutive rows over all banks.
template <bool Q4>
__global__ __launch_bounds__(256, 2) void k_gemm_q80(const ActQ8_0* __restrict__ act, int M, int nb,
                                                  const uint16_t* __restrict__ wd, const uint8_t* __restrict__ wqs,
                                                  int N, int tiles_m, int tiles_n, float* y, int64_t ldy,
                                                  const float* __restrict__ bias, const float* res, int64_t ldr) {
    __shared__ __align__(16) int8_t sa[2][kQBM * 128];
    __shared__ __align__(16) int8_t sb[2][kQBM * 128];
    __shared__ __align__(16) float sda[2][kQKC][kQBM];
    __shared__ float sdw[2][kQKC][kQBM];
    int mt, nt;
    xcd_tile(blockIdx.x, tiles_m, mt, nt);
    if (nt >= tiles_n) return;  // uniform: padding of the weight tiles to a multiple of 8
    const int m0 = mt * kQBM, n0 = nt * kQBM;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave & 1, wn = wave >> 1;
    const int l31 = lane & 31, h = lane >> 5;

    // staging roles: 16-byte piece p of rows pr + 32 i (activations, Q8_0 weights); block j of
    // rows jr + 64 i (scales, Q4_0 blocks).  Clamped rows and blocks (never used or stored).
    const int pr = tid >> 3, p = tid & 7, jr = tid >> 2, jb = tid & 3;
    v4i ra[2], rb[2];
    float rda;
    uint16_t rdw;
    auto stage_load = [&](int c0) {
        const int bp = min(c0 + (p >> 1), nb - 1), bj = min(c0 + jb, nb - 1);
#pragma unroll
        for (int i = 0; i < 2; ++i)
            ra[i] = *(const v4i*)(act[(int64_t)min(m0 + pr + 32 * i, M - 1) * nb + bp].qs + 16 * (p & 1));
        rda = act[(int64_t)min(m0 + jr, M - 1) * nb + bj].d;
        const int64_t row = (int64_t)min(n0 + jr, N - 1) * nb + bj;
        rdw = wd[row];
        if (Q4) {
            rb[0] = *(const v4i*)(wqs + row * 16);
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i)
                rb[i] = *(const v4i*)(wqs + ((int64_t)min(n0 + pr + 32 * i, N - 1) * nb + bp) * 32 + 16 * (p & 1));
        }
    };
    auto slot = [](int row, int piece) { return row * 128 + ((piece ^ ((row >> 1) & 7)) << 4); };
    auto stage_store = [&](int st) {
#pragma unroll
        for (int i = 0; i < 2; ++i) *(v4i*)(sa[st] + slot(pr + 32 * i, p)) = ra[i];
        sda[st][jb][jr] = rda;
        sdw[st][jb][jr] = f16_scale(rdw);
        if (Q4) {  // element j is the low nibble of byte j, j + 16 the high one
            v4i lo, hi;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                lo[t] = (int)nib_i8((uint32_t)rb[0][t]);
                hi[t] = (int)nib_i8((uint32_t)rb[0][t] >> 4);
            }
            *(v4i*)(sb[st] + slot(jr, 2 * jb)) = lo;
            *(v4i*)(sb[st] + slot(jr, 2 * jb + 1)) = hi;
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i) *(v4i*)(sb[st] + slot(pr + 32 * i, p)) = rb[i];
        }
    };

    float acc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
    const v16i zero = {};
    const int col = 32 * wn + l31;
    // One block in flight: its operands, then its dots and scales.
    struct Block {
        v4i a, b;
        v16i s;
        float da[16], dw;
    };
    auto read = [&](Block& k, int st, int j) {
        k.a = *(const v4i*)(sa[st] + slot(32 * wm + l31, 2 * j + h));
        k.b = *(const v4i*)(sb[st] + slot(col, 2 * j + h));
        k.dw = sdw[st][j][col];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 v = *(const float4*)&sda[st][j][32 * wm + 8 * q + 4 * h];
            k.da[4 * q] = v.x;
            k.da[4 * q + 1] = v.y;
            k.da[4 * q + 2] = v.z;
            k.da[4 * q + 3] = v.w;
        }
    };
    auto dots = [&](Block& k) { k.s = __builtin_amdgcn_mfma_i32_32x32x32_i8(k.a, k.b, zero, 0, 0, 0); };
    auto fold = [&](const Block& k) {
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = acc[i] + ((float)k.s[i] * k.dw) * k.da[i];
    };

    const int nc = (nb + kQKC - 1) / kQKC;
    stage_load(0);
    stage_store(0);
    stage_load(kQKC);
    lds_barrier();
    // While a block's dots run on the matrix cores, the block before it is folded (blocks
    // alternate between k0 and k1; the last block of a stage is folded behind the next one's
    // first reads).  The scheduling barriers keep that order.
    Block k0, k1;
    for (int c = 0; c < nc; ++c) {
        const int st = c & 1, kc = nb - c * kQKC;
        if (kc >= kQKC) {
            read(k0, st, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (c > 0) fold(k1);
            dots(k0);
            read(k1, st, 1);
            dots(k1);
            __builtin_amdgcn_sched_barrier(0);
            fold(k0);
            read(k0, st, 2);
            dots(k0);
            __builtin_amdgcn_sched_barrier(0);
            fold(k1);
            read(k1, st, 3);
            dots(k1);
            __builtin_amdgcn_sched_barrier(0);
            fold(k0);
        } else {
            if (c > 0) fold(k1);
            for (int j = 0; j < kc; ++j) {
                read(k1, st, j);
                dots(k1);
                if (j + 1 < kc) fold(k1);
            }
        }
        if (c + 1 < nc) {
            stage_store(st ^ 1);  // read last a stage ago, behind the barrier below
            stage_load((c + 2) * kQKC);
            lds_barrier();
        }
    }
    fold(k1);

    const int n = n0 + col;
    if (n >= N) return;
    const float bv = bias ? bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int m = m0 + 32 * wm + 8 * (i >> 2) + 4 * h + (i & 3);
        if (m >= M) continue;
        float v = bias ? acc[i] + bv : acc[i];
        if (res) v = res[(int64_t)m * ldr + n] + v;
        y[(int64_t)m * ldy + n] = v;
    }
}

// ---- in between: one wave per 16 x 16 tile ----------------------------------------------

static_assert(kMdActB == sizeof(ActQ8_0), "an activation block");

// The same chains in registers over 16 x 16 tiles (v_mfma_i32_16x16x32_i8, lanes as in the
// split kernel): a quarter of the per-block time, four times the tiles.  Stages of eight
// blocks are loaded two ahead into registers, because eight blocks take less time than a load.
// LDS: 16-byte piece p of row r at p ^ (r & 15), 256 bytes per row.
template <bool Q4>
__global__ __launch_bounds__(256, 2) void k_gemm_q80_mid(const ActQ8_0* __restrict__ act, int M, int nb,
                                                         const uint16_t* __restrict__ wd,
                                                         const uint8_t* __restrict__ wqs, int N, int tiles_m,
                                                         int tiles_n, float* y, int64_t ldy,
                                                         const float* __restrict__ bias, const float* res,
                                                         int64_t ldr) {
    __shared__ __align__(16) int8_t sa[2][kMdT * 256];
    __shared__ __align__(16) int8_t sb[2][kMdT * 256];
    __shared__ __align__(16) float sda[2][kMdKC][kMdT];
    __shared__ float sdw[2][kMdKC][kMdT];
    int mt, nt;
    xcd_tile(blockIdx.x, tiles_m, mt, nt);
    if (nt >= tiles_n) return;  // uniform: padding of the weight tiles to a multiple of 8
    const int m0 = mt * kMdT, n0 = nt * kMdT;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = 16 * (wave & 1), wn = 16 * (wave >> 1);
    const int r = lane & 15, g = lane >> 4;

    // staging roles: pieces p and p + 8 (blocks p / 2 and p / 2 + 4) of row pr; block jb of row
    // jr (scales, Q4_0 blocks)
    const int pr = tid >> 3, p = tid & 7, jr = tid >> 3, jb = tid & 7;
    const int rm = min(kMdT, M - m0), rn = min(kMdT, N - n0);
    auto rsrc = [](const void* p, uint32_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
    };
    constexpr uint32_t WB = Q4 ? 16 : 32;
    const __amdgpu_buffer_rsrc_t ars = rsrc(act + (int64_t)m0 * nb, (uint32_t)(rm * nb) * kMdActB);
    const __amdgpu_buffer_rsrc_t wrs = rsrc(wqs + (int64_t)n0 * nb * WB, (uint32_t)(rn * nb) * WB);
    const __amdgpu_buffer_rsrc_t drs = rsrc(wd + (int64_t)n0 * nb, (uint32_t)(rn * nb) * 2u);
    struct Regs {
        v4i a[2], b[2];
        float da;
        uint16_t dw;
    };
    // A thread's offsets stay; a stage only moves the scalar offset, and the stages at the row's end
    // (the last one, and the two loaded ahead of it) stop at the row's last eight blocks.
    const MidLoads o = mid_loads<Q4>(tid, rm, rn, nb);
    auto load = [&](Regs& k, int c0) {
        const uint32_t b = (uint32_t)mid_first(c0, nb);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            k.a[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(ars, o.a[i], b * kMdActB, 0));
            if (!Q4 || i == 0)
                k.b[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wrs, o.w[i], b * WB, 0));
        }
        k.da = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ars, o.da, b * kMdActB, 0));
        k.dw = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(drs, o.dw, b * 2u, 0);
    };
    auto slot = [](int row, int piece) { return row * 256 + ((piece ^ (row & 15)) << 4); };
    auto store = [&](const Regs& k, int st) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            *(v4i*)(sa[st] + slot(pr, p + 8 * i)) = k.a[i];
            if (!Q4) *(v4i*)(sb[st] + slot(pr, p + 8 * i)) = k.b[i];
        }
        sda[st][jb][jr] = k.da;
        sdw[st][jb][jr] = f16_scale(k.dw);
        if (Q4) {  // element j is the low nibble of byte j, j + 16 the high one
            v4i lo, hi;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                lo[t] = (int)nib_i8((uint32_t)k.b[0][t]);
                hi[t] = (int)nib_i8((uint32_t)k.b[0][t] >> 4);
            }
            *(v4i*)(sb[st] + slot(jr, 2 * jb)) = lo;
            *(v4i*)(sb[st] + slot(jr, 2 * jb + 1)) = hi;
        }
    };
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const v4i zero = {};
    struct Block {
        long a, b;
        float4 da;
        float dw;
    };
    auto read = [&](Block& k, int st, int j) {  // lane (r, g): elements 8g .. 8g + 7 of both rows
        k.a = *(const long*)(sa[st] + slot(wm + r, 2 * j + (g >> 1)) + 8 * (g & 1));
        k.b = *(const long*)(sb[st] + slot(wn + r, 2 * j + (g >> 1)) + 8 * (g & 1));
        k.da = *(const float4*)&sda[st][j][wm + 4 * g];
        k.dw = sdw[st][j][wn + r];
    };
    auto dots = [&](const Block& k) { return __builtin_amdgcn_mfma_i32_16x16x32_i8(k.a, k.b, zero, 0, 0, 0); };
    auto fold = [&](const Block& k, const v4i& s) {
        acc[0] = acc[0] + ((float)s[0] * k.dw) * k.da.x;
        acc[1] = acc[1] + ((float)s[1] * k.dw) * k.da.y;
        acc[2] = acc[2] + ((float)s[2] * k.dw) * k.da.z;
        acc[3] = acc[3] + ((float)s[3] * k.dw) * k.da.w;
    };
    // Four blocks' operands are read and multiplied together, and the next four read while
    // they are folded: a wave often has its SIMD to itself, and block by block it waited for
    // LDS and the matrix cores at each (896 x 4864 at 226 rows 24.9 us, now 21.3).
    auto compute = [&](int st, int c) {
        const int kc = nb - c * kMdKC;
        if (kc >= kMdKC) {
            Block k[4], n[4];
            v4i s[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) read(k[j], st, j);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] = dots(k[j]);
#pragma unroll
            for (int j = 0; j < 4; ++j) read(n[j], st, 4 + j);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 4; ++j) fold(k[j], s[j]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] = dots(n[j]);
#pragma unroll
            for (int j = 0; j < 4; ++j) fold(n[j], s[j]);
        } else {
            const int c0 = c * kMdKC, slot0 = c0 - mid_first(c0, nb);
            for (int j = 0; j < kc; ++j) {
                Block k;
                read(k, st, slot0 + j);
                fold(k, dots(k));
            }
        }
    };

    const int nc = (nb + kMdKC - 1) / kMdKC;
    Regs r0, r1;
    load(r0, 0);
    load(r1, kMdKC);
    store(r0, 0);
    // r1's loads stay ahead of r0's: interleaved, a wait for one stage's takes the other's too (the
    // 226-row CosyVoice2 prompt 2043 us, now 2024)
    __builtin_amdgcn_sched_barrier(0);
    load(r0, 2 * kMdKC);
    lds_barrier();
    for (int c = 0;; c += 2) {
        compute(0, c);
        if (c + 1 >= nc) break;  // uniform
        store(r1, 1);            // stage buffers: read last a stage ago, behind a barrier
        load(r1, (c + 3) * kMdKC);
        lds_barrier();
        compute(1, c + 1);
        if (c + 2 >= nc) break;
        store(r0, 0);
        load(r0, (c + 4) * kMdKC);
        lds_barrier();
    }

    const int n = n0 + wn + r;
    if (n >= N) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + wm + 4 * g + i;
        if (m >= M) continue;
        float v = bias ? acc[i] + bias[n] : acc[i];
        if (res) v = res[(int64_t)m * ldr + n] + v;
        y[(int64_t)m * ldy + n] = v;
    }
}

template <bool Q4>
static hipError_t gemm_q80_dispatch(const QWeight& w, const ActQ8_0* act, int m, float* y, int64_t ldy,
                                    const float* bias, const float* res, int64_t ldr, hipStream_t s) {
    const int nb = (int)w.nb, N = (int)w.n;
    const uint16_t* wd = (const uint16_t*)w.hdr;
    auto tiles = [](int64_t v, int t) { return (int)((v + t - 1) / t); };
#define SXQ_Q80(K, THREADS, BM, BN, LDS)                                                                     \
    do {                                                                                                     \
        const int tm = tiles(m, BM), tn = tiles(N, BN);                                                      \
        static const hipError_t attr = hipFuncSetAttribute(                                                  \
            (const void*)(K), hipFuncAttributeMaxDynamicSharedMemorySize, (int)(LDS));                       \
        if (attr != hipSuccess) return attr;                                                                 \
        hipLaunchKernelGGL((K), dim3((unsigned)(tiles(tn, 8) * 8 * tm)), dim3(THREADS), LDS, s, act, m, nb, wd, w.qs, N, \
                           tm, tn, y, ldy, bias, res, ldr);                                                  \
        return hipGetLastError();                                                                            \
    } while (0)
    // The kernel by the number of 16 x 16 tiles, T, and of 64 x 64 tiles, T64 (us with the
    // activation quantizer's launch, in a graph):
    //  T <= 256, a workgroup per CU: the split kernel with 32-block chunks (split 32 / split 16 /
    //  mid: 896 x 4864 at 64 rows, T = 224: 12.0 / 12.8 / 18.8, at 65 rows, T = 280: 18.8 / 16.4 /
    //  18.7; 2048 x 1024 at 32 rows, T = 256: 5.8 / 6.1 / 7.7, at 33 rows, T = 384: 7.8 / 7.0 / 7.8).
    //  T <= 512, two per CU: with 16-block chunks (split 16 / mid: 2560 x 9728 at 48 rows, T = 480:
    //  27.2 / 32.4, at 49 rows, T = 640: 34.9 / 32.6; 896 x 4864 at 144 rows, T = 504: 17.6 / 19.7, at
    //  145 rows, T = 560: 21.5 / 19.6), and up to three per CU for 16 rows, where half of each of
    //  mid's row tiles is padding (12288 x 896, T = 768: 8.0 / 8.9; 16384 x 2560, T = 1024: 16.2 / 15.7).
    //  T64 < 400, or one row tile of 32: mid (mid / 64 x 64: 4864 x 896 at 226 rows, T64 = 304: 14.9 /
    //  16.0, at 300 rows, 380: 16.9 / 16.3; 6564 x 896 at 200 rows, 412: 16.6 / 16.2; 2560 x 9728 at 600
    //  rows, 400: 99 / 107, at 640 rows: 114 / 107; 1152 x 896 at 1500 rows, 432: 22.8 / 22.1; 151936 x
    //  896 at 32 rows 43.0 / 49.5, at 33 rows 71.7 / 49.7); from there on 64 x 64.
    // One wave per 32 x 64 tile was never ahead of 32 x 32 (9728 x 896 at 1024 rows: 70.8 against
    // 67.5), nor the split kernel with 32 rows per workgroup ahead of both others.
    const int64_t T = (int64_t)tiles(m, 16) * tiles(N, kSpN);
    if (T <= 256) SXQ_Q80((k_gemm_q80_split<Q4, 4>), 512, 16, kSpN, (SplitShape<Q4, 4>::lds));
    if (T <= (m <= 16 ? 768 : 512)) SXQ_Q80((k_gemm_q80_split<Q4, 2>), 512, 16, kSpN, (SplitShape<Q4, 2>::lds));
    if (m <= kMdT || (int64_t)tiles(m, kQBM) * tiles(N, kQBM) < 400) SXQ_Q80((k_gemm_q80_mid<Q4>), 256, kMdT, kMdT, 0);
    SXQ_Q80((k_gemm_q80<Q4>), 256, kQBM, kQBM, 0);
#undef SXQ_Q80
}

hipError_t launch_gemm_q80(const QWeight& w, const void* act, int m, float* y, int64_t ldy, const float* bias,
                           const float* res, int64_t ldr, hipStream_t s) {
    if ((w.dtype != kQ8_0 && w.dtype != kQ4_0) || m <= 0) return hipErrorInvalidValue;
    return w.dtype == kQ8_0 ? gemm_q80_dispatch<false>(w, (const ActQ8_0*)act, m, y, ldy, bias, res, ldr, s)
                            : gemm_q80_dispatch<true>(w, (const ActQ8_0*)act, m, y, ldy, bias, res, ldr, s);
}

}  // namespace sxq
