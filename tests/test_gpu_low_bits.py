"""Low bits of activations and weights on the fp16 matrix-core kernels, whose
operands are split into parts: the product of the two low parts, elements far
below others that share their exponent, and subnormal tokens."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from forge_amd import formats as F
from forge_amd import ops, synth
from test_gpu_parity import dev_weight

pytestmark = pytest.mark.gpu
KQ = [F.Q4_K, F.Q5_K, F.Q6_K]
ALL = KQ + [F.Q4_0, F.Q4_1, F.Q8_0, F.Q5_0, F.Q5_1, F.IQ4_NL]


def run(dtype, w, x, N, K):
    return ops.matmul_transB(torch.from_numpy(x).cuda(), dev_weight(dtype, w, N, K)).cpu().numpy()


def rel(dtype, w, x, N, K):
    ref = oracle.matmul_f64(dtype, x, w, N, K)
    return np.linalg.norm(run(dtype, w, x, N, K) - ref) / np.linalg.norm(ref)


def zero_first_64(dtype, w, N):
    """Weights that are zero in the first 64 elements of every 256."""
    f = F.fmt(dtype)
    b = w.reshape(N, -1, f.block_bytes).copy()
    if dtype == F.Q6_K:
        b[:, :, 192:196] = 0
    elif dtype in (F.Q4_K, F.Q5_K):
        b[:, :, [4, 5, 8, 9]] &= 0xC0
    else:
        for i in (0, 1):
            b[:, i::8, 0:4 if dtype in (F.Q4_1, F.Q5_1) else 2] = 0
    return b.reshape(N, -1)


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


# an element of 2^27 times the others in every super-block, in the 64 elements
# whose weights are zero: the others' bits are theirs
@pytest.mark.parametrize("dtype,M", [(d, 20) for d in ALL] + [(F.Q5_K, 40)])
def test_small_elements_beside_large_ones(dtype, M):
    N, K = 130, 1024
    w = zero_first_64(dtype, synth.make_weights(dtype, N, K, seed=3), N)
    x = synth.make_x(M, K, seed=4)
    x[:, 5::256] = np.float32(2.0 ** 27)
    assert rel(dtype, w, x, N, K) <= 1e-6


# such an element in a super-block of zero weights, minima of zero: the sums that
# centre the codes keep the bits of the other super-blocks.  Q4_K prefill has one
# exponent per token: its elements keep 2^-39 of the largest, 2^-39 2^19 of the
# others, 1e-6 of the result at most; sums in fp16 hi + lo kept 2^-34
@pytest.mark.parametrize("dtype,log2", [(F.Q4_K, 19), (F.Q5_K, 20), (F.Q5_K, 60)])
def test_small_super_blocks_beside_large_ones(dtype, log2):
    N, K, M = 130, 1024, 40
    w = synth.make_weights(dtype, N, K, seed=7).reshape(N, -1, F.fmt(dtype).block_bytes)
    w[:, 1, 0:2] = 0  # d
    w[:, :, 2:4] = 0  # dmin
    x = synth.make_x(M, K, seed=8)
    x[:, 256 + 77] = np.float32(2.0 ** log2)
    assert rel(dtype, w.reshape(N, -1), x, N, K) <= 1e-6


# tokens of subnormal numbers against weights large enough for normal results
@pytest.mark.parametrize("M", [20, 40])
@pytest.mark.parametrize("dtype", KQ)
def test_subnormal_tokens(dtype, M):
    N, K = 70, 512
    f = F.fmt(dtype)
    w = synth.make_weights(dtype, N, K, seed=5).reshape(N, -1, f.block_bytes)
    at = 208 if dtype == F.Q6_K else 0
    w[:, :, at:at + 2] = np.frombuffer(np.float16(30000.0).tobytes(), dtype=np.uint8)
    x = (np.random.default_rng(6).integers(-300, 301, (M, K)) * 2.0 ** -149).astype(np.float32)
    assert rel(dtype, w.reshape(N, -1), x, N, K) <= 1e-6
