"""Several matrices in one band-kernel launch (5..16 tokens, unsplit K): the
same bits as one call per matrix, at ragged rows, empty matrices and each
format's tile counts."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from forge_amd import formats as F
from forge_amd import ops, synth
from helpers import assert_close_silu_mul
from test_gpu_parity import dev_weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", sorted(F.FORMATS))
@pytest.mark.parametrize("M,K,ns", [(5, 256, (17, 1, 16)), (16, 2048, (2048, 256, 256)),
                                    (8, 4096, (5000, 0, 33)), (11, 1024, (0, 9000, 15))])
def test_qkv_bits(dtype, M, K, ns):
    x = torch.from_numpy(synth.make_x(M, K, seed=M)).cuda()
    W = [dev_weight(dtype, synth.make_weights(dtype, n, K, 40 + i), n, K) for i, n in enumerate(ns)]
    y = ops.fused_qkv(x, *W)
    assert torch.equal(y, torch.cat([ops.matmul_transB(x, w) for w in W], dim=1))


@pytest.mark.parametrize("dtype", sorted(F.FORMATS))
@pytest.mark.parametrize("M,N,K", [(5, 1, 256), (16, 33, 512), (8, 5632, 2048), (9, 8200, 768)])
def test_gate_up(dtype, M, N, K):
    wg, wu = (synth.make_weights(dtype, N, K, s) for s in (50, 51))
    x = synth.make_x(M, K, seed=M) * np.float32(1e-2)
    xd = torch.from_numpy(x).cuda()
    G, U = dev_weight(dtype, wg, N, K), dev_weight(dtype, wu, N, K)
    y = ops.ffn_up_fused(xd, G, U)
    g, u = (oracle.matmul_f64(dtype, x, w, N, K) for w in (wg, wu))
    wm = max(float(np.max(np.abs(oracle.dequant(dtype, w, N, K)))) for w in (wg, wu))
    assert_close_silu_mul(y.cpu().numpy(), g, u, x, wm, f"{dtype} {M}x{N}x{K}")
    if dtype == F.Q5_1:  # the band kernel takes it from K = 14336 only
        return
    ref = torch.nn.functional.silu(ops.matmul_transB(xd, G)) * ops.matmul_transB(xd, U)
    torch.testing.assert_close(y, ref, rtol=2e-6, atol=1e-9)  # only the two SiLUs differ
