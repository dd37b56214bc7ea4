"""Low bits of activations and weights on the fp16 matrix-core kernels, whose
operands are split into parts: the product of the two low parts."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from forge_amd import formats as F
from forge_amd import ops, synth
from test_gpu_parity import dev_weight

pytestmark = pytest.mark.gpu


def run(dtype, w, x, N, K):
    return ops.matmul_transB(torch.from_numpy(x).cuda(), dev_weight(dtype, w, N, K)).cpu().numpy()


# Q6_K, 17..32 tokens: x = hi + lo and sc (q - 32) = 2057 = hi + lo in fp16, both
# low parts 2^-11 of the whole, so their product is 2^-22 of the result.  One
# product per sum and d a power of two leave two fp32 roundings.
def test_product_of_the_low_parts():
    N, K, M = 64, 512, 32
    w = np.zeros((N, K // 256, 210), dtype=np.uint8)
    code = 17 + 32  # (q - 32) = 17, sc = 121
    w[:, :, 0:128] = (code & 15) * 0x11
    w[:, :, 128:192] = (code >> 4) * 0x55
    w[:, :, 192:208] = 121
    w[:, :, 208:210] = np.frombuffer(np.float16(2.0 ** -12).tobytes(), dtype=np.uint8)
    w = w.reshape(N, -1)
    x = np.zeros((M, K), dtype=np.float32)
    v = np.float32(1 + 2.0 ** -11 - 2.0 ** -21)
    x[np.arange(M), np.arange(M) * 15 + 7] = v
    exact = float(v) * 2057 * 2.0 ** -12
    assert np.abs(run(F.Q6_K, w, x, N, K) - exact).max() <= 3 * 2.0 ** -24 * exact
