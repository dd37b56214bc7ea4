"""The prefill kernels' activation operands and token tiles: rows at the edges
of what the preparation keeps in registers (32768 elements up to 128 tokens,
8192 and 20480 above), tokens that end in the first and in the second 32 of a
wave's 64."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from forge_amd import formats as F
from forge_amd import ops, synth
from helpers import assert_close
from test_gpu_parity import dev_weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [F.Q8_0, F.Q5_1, F.Q6_K, F.Q5_K])
@pytest.mark.parametrize("M,N,K", [(33, 40, 32768), (40, 33, 33024), (128, 64, 8448), (129, 64, 8192),
                                   (132, 40, 8448), (161, 33, 20480), (193, 31, 20736), (97, 70, 256)])
def test_row_lengths(dtype, M, N, K):
    w = synth.make_weights(dtype, N, K, seed=M)
    x = synth.make_x(M, K, seed=K + 3)
    x[0, -1] = np.float32(1e4)  # the largest element in the row's last piece
    x[M - 1] *= np.float32(1e-12)
    y = ops.matmul_transB(torch.from_numpy(x).cuda(), dev_weight(dtype, w, N, K)).cpu().numpy()
    deq_max = np.array([float(np.max(np.abs(oracle.dequant(dtype, w, N, K))))])
    for rows in (slice(0, M - 1), slice(M - 1, M)):  # by magnitude
        assert_close(y[rows], oracle.matmul_f64(dtype, x[rows], w, N, K), x[rows], deq_max, f"{dtype} {M}x{N}x{K}")
