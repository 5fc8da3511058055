// sxq_q80_stage.h -- which bytes a thread of k_gemm_q80_mid loads for an LDS stage.  Plain
// constant expressions, so that the CPU can enumerate every load of a shape.
#pragma once
#include <cstdint>

namespace sxq {

constexpr int kMdT = 32;          // rows and weight rows per workgroup: 2 x 2 waves
constexpr int kMdKC = 8;          // blocks per LDS stage
constexpr uint32_t kMdActB = 48;  // bytes of an activation block: 32 quants, then the f32 scale

// The first block loaded by the stage that begins at block c0 of nb: the stages at the end of the
// row load its last eight blocks, and block c0 + j is then in slot c0 - mid_first(c0, nb) + j.
constexpr int mid_first(int c0, int nb) {
    const int full = nb > kMdKC ? nb - kMdKC : 0;
    return c0 < full ? c0 : full;
}

// Byte offsets, from the tile's first row and the stage's first block, of a thread's loads:
// activation and Q8_0 weight quants as two 16-byte pieces each (slots p / 2 and p / 2 + 4 of row
// tid / 8, p = tid mod 8), an activation scale, a Q4_0 block (w[0]) and a weight scale (slot p of
// that row).  rm, rn: the tile's rows that exist; nb: blocks per row.  A row, or a slot of a row
// of fewer than eight blocks, that does not exist is replaced by the last one that does, so
// every load stays inside the operands by itself; what it gives is never added or stored.
struct MidLoads {
    uint32_t a[2], da, w[2], dw;
};
template <bool Q4>
constexpr MidLoads mid_loads(int tid, int rm, int rn, int nb) {
    const int row = tid >> 3, p = tid & 7, last = nb - 1;
    const uint32_t ra = (uint32_t)((row < rm ? row : rm - 1) * nb), rw = (uint32_t)((row < rn ? row : rn - 1) * nb);
    const uint32_t b0 = (uint32_t)((p >> 1) < last ? p >> 1 : last);
    const uint32_t b1 = (uint32_t)((p >> 1) + 4 < last ? (p >> 1) + 4 : last);
    const uint32_t bj = (uint32_t)(p < last ? p : last);
    const uint32_t half = 16u * (uint32_t)(p & 1);
    MidLoads o = {};
    o.a[0] = (ra + b0) * kMdActB + half;
    o.a[1] = (ra + b1) * kMdActB + half;
    o.da = (ra + bj) * kMdActB + 32u;
    o.w[0] = Q4 ? (rw + bj) * 16u : (rw + b0) * 32u + half;
    o.w[1] = Q4 ? o.w[0] : (rw + b1) * 32u + half;
    o.dw = (rw + bj) * 2u;
    return o;
}

}  // namespace sxq
