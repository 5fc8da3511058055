"""GPU kernels at the edges of their tiles: remainders, unaligned pointers, the smallest and
largest sizes each dispatch rule sends to them, against the CPU oracle."""
import ctypes

import numpy as np
import pytest
import torch

from syrinx_amd import GgmlDType, QMatMul, QTensor
from syrinx_amd._lib import check, lib

pytestmark = pytest.mark.gpu

G = GgmlDType


@pytest.fixture(scope="module")
def cuda():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm GPU (torch.cuda.is_available() is False)")
    return torch.device("cuda:0")


def _rows(n, k, seed):
    """Normal rows with blocks of zeros, ties, tiny and huge values, infinities and NaN."""
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


# (n, k, m): weight tiles of 16 / 64 / 128 rows and row tiles of 16 / 32 / 64 with remainders,
# block counts below, at and past a chunk (4, 8, 16, 32 blocks), each kernel of the dispatch
Q80_SHAPES = [(1, 32, 5), (17, 320, 16), (16, 1024, 17), (130, 1056, 33), (896, 4864, 8), (77, 992, 64), (200, 160, 65),
              (1152, 896, 226), (2048, 1024, 500), (4100, 96, 130), (896, 4864, 226), (9728, 896, 50), (64, 2080, 300)]


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
