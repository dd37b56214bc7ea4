"""Q4_K and Q5_K prefill with the sub-block scales in the weight operand:
partial token and row tiles, K of one super-block and of an odd number per
split, codes, scales and minima at their extremes, every bias form."""
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


def check(dtype, w, x, N, K, y, what):
    deq_max = float(np.max(np.abs(oracle.dequant(dtype, w, N, K))))
    assert_close(y, oracle.matmul_f64(dtype, x, w, N, K), x, np.array([deq_max]), what)


@pytest.mark.parametrize("dtype", [F.Q4_K, F.Q5_K])
@pytest.mark.parametrize("M,N,K", [(33, 1, 256), (64, 257, 768), (65, 31, 2816), (96, 255, 1024),
                                   (129, 256, 512), (77, 300, 18944), (160, 513, 3584)])
def test_tile_edges(dtype, M, N, K):
    w = synth.make_weights(dtype, N, K, seed=M + N)
    x = synth.make_x(M, K, seed=K + 1)
    x[M // 2] = 0.0
    x[1] *= np.float32(1e20)
    x[2] *= np.float32(1e-20)
    W, xd = dev_weight(dtype, w, N, K), torch.from_numpy(x).cuda()
    y = ops.matmul_transB(xd, W)
    for rows in (slice(0, 1), slice(1, 2), slice(2, 3), slice(3, M)):  # by magnitude
        check(dtype, w, x[rows], N, K, y[rows].cpu().numpy(), f"{dtype} {M}x{N}x{K} {rows}")
    assert not y[M // 2].any()
    b1 = torch.from_numpy(synth.make_x(1, N, seed=5).reshape(N)).cuda()
    b2 = torch.from_numpy(synth.make_x(M, N, seed=6)).cuda()
    assert torch.equal(ops.matmul_transB(xd, W, b2)[3:], (y + b2)[3:])
    assert torch.equal(ops.matmul_transB(xd, W, b1)[3:], (y + b1)[3:])


@pytest.mark.parametrize("dtype", [F.Q4_K, F.Q5_K])
def test_extreme_codes_and_scales(dtype):
    # every (code extreme, sub-block scale, minimum): rows of all-zero and
    # all-one code bits with scale bytes 0x00, 0x3F, 0xFF and random ones
    N, K, M = 64, 512, 40
    f = F.fmt(dtype)
    w = synth.make_weights(dtype, N, K, seed=9).reshape(N, -1, f.block_bytes)
    body = slice(16, f.block_bytes)
    for r in range(N):
        if r % 4 < 2:
            w[r, :, body] = 255 * (r % 2)
        if r % 8 < 6:
            w[r, :, 4:16] = (0x00, 0x3F, 0xFF)[(r % 8) // 2]
    x = synth.make_x(M, K, seed=10)
    y = ops.matmul_transB(torch.from_numpy(x).cuda(), dev_weight(dtype, w.reshape(N, -1), N, K))
    check(dtype, w.reshape(N, -1), x, N, K, y.cpu().numpy(), "extremes")
    # a one-hot token (an exact power of two) reproduces its column's value
    # within the two fp32 roundings of d D - dmin Dm
    deq = oracle.dequant(dtype, w.reshape(N, -1), N, K).reshape(N, K)
    hot = np.zeros((M, K), dtype=np.float32)
    cols = np.arange(M) * 12 + 3
    hot[np.arange(M), cols] = 1.0
    y = ops.matmul_transB(torch.from_numpy(hot).cuda(), dev_weight(dtype, w.reshape(N, -1), N, K))
    d = w[:, :, 0:4].copy().view(np.float16).astype(np.float64)  # d, dmin
    scale = 63 * (31 * np.abs(d[..., 0]) + np.abs(d[..., 1]))[:, cols // 256].T
    assert (np.abs(y.cpu().numpy() - deq[:, cols].T) <= 2.0 ** -23 * scale).all()


def test_q5k_noalloc_beyond_the_prefill_plan():
    # 16 K-splits need 65 MiB of the fixed 64: fewer tokens at a time
    from forge_amd import _lib

    M, N, K = 2040, 256, 4096
    w = synth.make_weights(F.Q5_K, N, K, seed=21)
    x = torch.from_numpy(synth.make_x(M, K, seed=22)).cuda()
    W = dev_weight(F.Q5_K, w, N, K)
    y = torch.empty((M, N), device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    assert _lib.lib().fq_matmul_transB_noalloc(F.Q5_K, x.data_ptr(), W.data.data_ptr(), None, 0, 0,
                                               y.data_ptr(), M, K, N, st) == 0
    deq = torch.from_numpy(oracle.dequant(F.Q5_K, w, N, K).reshape(N, K)).cuda().double()
    ref = x.double() @ deq.T
    for got in (y, ops.matmul_transB(x, W)):
        assert float((got.double() - ref).norm() / ref.norm()) <= 1e-5
    assert torch.equal(y, ops.matmul_transB(x, W))
