"""Every load of k_gemm_q80_mid's LDS stages, enumerated on the CPU from the offsets the kernel
uses (csrc/sxq_q80_stage.h): each stays inside the operands, whatever the buffer's range check
does, and each row and block that exists is loaded from its own place."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include "sxq_q80_stage.h"
using namespace sxq;

// One load: `size` bytes at `at` of an operand of `rows` rows of nb blocks of B bytes; where row
// and block exist it must be byte `in` of that block.
static bool ok(uint32_t at, uint32_t size, int rows, int nb, uint32_t B, int row, int block, uint32_t in) {
    if ((uint64_t)at + size > (uint64_t)rows * nb * B) return false;
    return row >= rows || block >= nb || at == (uint32_t)(row * nb + block) * B + in;
}

template <bool Q4>
static bool shape(int rm, int rn, int nb) {
    for (int c0 = 0; c0 < nb + 4 * kMdKC; c0 += kMdKC) {  // the kernel loads up to two stages past the last
        const int first = mid_first(c0, nb);
        // every block of the stage has a slot of its own among the eight
        if (c0 < nb && (first > c0 || (c0 + kMdKC < nb ? c0 + kMdKC : nb) > first + kMdKC)) return false;
        for (int tid = 0; tid < 256; ++tid) {
            const MidLoads o = mid_loads<Q4>(tid, rm, rn, nb);
            const int row = tid >> 3, p = tid & 7;
            const uint32_t h = 16u * (p & 1), wb = Q4 ? 16 : 32;
            for (int i = 0; i < 2; ++i) {
                const int b = first + p / 2 + 4 * i;
                if (!ok(o.a[i] + first * kMdActB, 16, rm, nb, kMdActB, row, b, h)) return false;
                if (!Q4 && !ok(o.w[i] + first * wb, 16, rn, nb, wb, row, b, h)) return false;
            }
            if (!ok(o.da + first * kMdActB, 4, rm, nb, kMdActB, row, first + p, 32)) return false;
            if (Q4 && !ok(o.w[0] + first * wb, 16, rn, nb, wb, row, first + p, 0)) return false;
            if (!ok(o.dw + first * 2u, 2, rn, nb, 2, row, first + p, 0)) return false;
        }
    }
    return true;
}

int main() {
    const int rows[] = {1, 2, 18, 31, 32};
    for (int nb = 1; nb <= 40; ++nb)
        for (int rm : rows)
            for (int rn : rows)
                if (!shape<false>(rm, rn, nb) || !shape<true>(rm, rn, nb)) {
                    std::printf("rows %d, weight rows %d, blocks %d: a load outside or misplaced\n", rm, rn, nb);
                    return 1;
                }
    std::printf("ok\n");
}
"""


def test_mid_stage_loads_stay_inside_the_operands(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not installed")
    src, exe = tmp_path / "stage.cpp", tmp_path / "stage"
    src.write_text(DRIVER)
    subprocess.run([gxx, "-std=c++17", "-O1", "-I", os.path.join(ROOT, "syrinx_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
