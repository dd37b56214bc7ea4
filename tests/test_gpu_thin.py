"""Small batches with the token operands shared by a work-group (24 to 48 MiB
and more, or 17..32 tokens; gate/up pairs of 2..4 tokens): partial row tiles, one
super-block, odd counts of them over two wave groups and K-splits, both token
tiles partly filled, offset bases, gate/up pairs and concatenated results."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from forge_amd import formats as F
from forge_amd import ops, synth
from helpers import assert_close, assert_close_silu_mul
from test_gpu_parity import dev_weight

pytestmark = pytest.mark.gpu
KQ = [F.Q4_K, F.Q5_K, F.Q6_K]
ALL = KQ + [F.Q4_0, F.Q4_1, F.Q8_0, F.Q5_0, F.Q5_1, F.IQ4_NL]


def wmax(dtype, ws, K):
    return max(float(np.max(np.abs(oracle.dequant(dtype, w[:2048], min(len(w), 2048), K)))) for w in ws)


@pytest.mark.parametrize("dtype", ALL)
@pytest.mark.parametrize("M,N,K", [(17, 1, 256), (32, 127, 512), (18, 300, 768), (31, 129, 2816),
                                   (24, 4100, 1024), (32, 33, 18944),
                                   (4, 24001, 2048), (5, 9000, 5888), (16, 3584, 18944),
                                   (9, 65537, 1024)])
def test_shapes(dtype, M, N, K):
    w = synth.make_weights(dtype, N, K, seed=M + N)
    x = synth.make_x(M, K, seed=K + M)
    x[M - 1, :256] = 0.0
    x[0] *= np.float32(1e18)
    x[1] *= np.float32(1e-18)
    xd = torch.from_numpy(x).cuda()
    W = dev_weight(dtype, w, N, K)
    y = ops.matmul_transB(xd, W)
    wm = wmax(dtype, [w], K)
    ref = oracle.matmul_f64(dtype, x, w, N, K)
    for r in (slice(0, 1), slice(1, 2), slice(2, M)):
        assert_close(y[r].cpu().numpy(), ref[r], x[r], np.array([wm]), f"{dtype} {M}x{N}x{K}")
    assert torch.equal(y, ops.matmul_transB(xd, W))  # deterministic
    b1 = torch.from_numpy(synth.make_x(1, N, seed=5).reshape(N)).cuda()
    b2 = torch.from_numpy(synth.make_x(M, N, seed=6)).cuda()
    tol = dict(rtol=1e-6, atol=1e-6 * float(y[2:].abs().max()))
    torch.testing.assert_close(ops.matmul_transB(xd, W, b1)[2:], (y + b1)[2:], **tol)
    torch.testing.assert_close(ops.matmul_transB(xd, W, b2)[2:], (y + b2)[2:], **tol)
    if dtype == F.Q6_K:  # every row's shift changes, no value does
        assert torch.equal(ops.matmul_transB(xd, dev_weight(dtype, w, N, K, 2)), y)


@pytest.mark.parametrize("dtype", ALL)
@pytest.mark.parametrize("M,N,K", [(17, 1, 256), (32, 65, 768), (20, 300, 2048), (2, 11008, 4096),
                                   (8, 14336, 4096), (16, 18945, 3584), (3, 4096, 14336),
                                   (4, 33, 512), (2, 500, 1024)])
def test_gate_up_pair(dtype, M, N, K):
    wg, wu = (synth.make_weights(dtype, N, K, s) for s in (50, 51))
    x = synth.make_x(M, K, seed=M) * np.float32(1e-2)
    y = ops.ffn_up_fused(torch.from_numpy(x).cuda(), dev_weight(dtype, wg, N, K),
                         dev_weight(dtype, wu, N, K))
    g, u = (oracle.matmul_f64(dtype, x, w, N, K) for w in (wg, wu))
    assert_close_silu_mul(y.cpu().numpy(), g, u, x, wmax(dtype, [wg, wu], K), f"{dtype} {M}x{N}x{K}")


@pytest.mark.parametrize("dtype", ALL)
@pytest.mark.parametrize("M,K,ns", [(17, 256, (257, 64, 1)), (32, 2048, (1, 300, 255)),
                                    (20, 512, (0, 96, 33)), (25, 1280, (31, 0, 256))])
def test_qkv(dtype, M, K, ns):
    ws = [synth.make_weights(dtype, n, K, 40 + i) for i, n in enumerate(ns)]
    x = synth.make_x(M, K, seed=M)
    y = ops.fused_qkv(torch.from_numpy(x).cuda(), *(dev_weight(dtype, w, n, K) for w, n in zip(ws, ns)))
    real = [w for w in ws if len(w)]
    ref = np.concatenate([oracle.matmul_f64(dtype, x, w, len(w), K) for w in real], axis=1)
    assert_close(y.cpu().numpy(), ref, x, np.array([wmax(dtype, real, K)]), f"qkv {dtype} {ns}")


@pytest.mark.parametrize("dtype", KQ)
def test_extreme_codes_and_scales(dtype):
    # codes and scales at both ends, and one-hot tokens, whose outputs are
    # the column's values within the fold's fp32 roundings
    N, K, M = 64, 768, 32
    f = F.fmt(dtype)
    w = synth.make_weights(dtype, N, K, seed=9).reshape(N, -1, f.block_bytes)
    at = slice(192, 208) if dtype == F.Q6_K else slice(4, 16)
    codes = slice(0, 192) if dtype == F.Q6_K else slice(16, f.block_bytes)
    for r in range(N):
        if r % 4 < 2:
            w[r, :, codes] = 255 * (r % 2)
        if r % 8 < 6:
            w[r, :, at] = (0x80, 0x7F, 0x3F)[(r % 8) // 2] if dtype == F.Q6_K else (0x00, 0x3F, 0xFF)[(r % 8) // 2]
    w = w.reshape(N, -1)
    x = synth.make_x(M, K, seed=10)
    W = dev_weight(dtype, w, N, K)
    y = ops.matmul_transB(torch.from_numpy(x).cuda(), W)
    assert_close(y.cpu().numpy(), oracle.matmul_f64(dtype, x, w, N, K), x, np.array([wmax(dtype, [w], K)]), "extremes")
    deq = oracle.dequant(dtype, w, N, K).reshape(N, K)
    hot = np.zeros((M, K), dtype=np.float32)
    cols = np.arange(M) * 23 + 5
    hot[np.arange(M), cols] = 1.0
    y = ops.matmul_transB(torch.from_numpy(hot).cuda(), W).cpu().numpy()
    if dtype == F.Q6_K:
        np.testing.assert_array_equal(y + np.float32(0.0), deq[:, cols].T + np.float32(0.0))
    else:
        d = w.reshape(N, -1, f.block_bytes)[:, :, 0:4].copy().view(np.float16).astype(np.float64)
        scale = 63 * (31 * np.abs(d[..., 0]) + np.abs(d[..., 1]))[:, cols // 256].T
        assert (np.abs(y - deq[:, cols].T) <= 2.0 ** -22 * scale).all()


# More row tiles than CUs: a work-group's range of steps runs over the ends of
# several tiles, whole ones and parts, odd step counts over two wave groups,
# from one matrix into the next
@pytest.mark.parametrize("dtype", [F.Q4_K, F.Q6_K, F.Q5_1, F.Q8_0])
@pytest.mark.parametrize("M,K,ns", [(21, 256, (70001,)), (32, 768, (40000,)), (18, 1280, (33333,)),
                                    (27, 768, (17001, 130, 16400))])
def test_ranges_over_tiles(dtype, M, K, ns):
    ws = [synth.make_weights(dtype, n, K, 70 + i) for i, n in enumerate(ns)]
    x = synth.make_x(M, K, seed=M)
    xd, Ws = torch.from_numpy(x).cuda(), [dev_weight(dtype, w, n, K) for w, n in zip(ws, ns)]
    y = ops.matmul_transB(xd, Ws[0]) if len(ns) == 1 else ops.fused_qkv(xd, *Ws)
    ref = np.concatenate([oracle.matmul_f64(dtype, x, w, len(w), K) for w in ws], axis=1)
    assert_close(y.cpu().numpy(), ref, x, np.array([wmax(dtype, ws, K)]), f"{dtype} {M} {ns} {K}")


@pytest.mark.parametrize("dtype", [F.Q4_K, F.Q6_K, F.Q5_1, F.Q8_0])
@pytest.mark.parametrize("M,N,K", [(3, 20003, 1280), (4, 40000, 256), (30, 20100, 768)])
def test_pair_ranges_over_tiles(dtype, M, N, K):
    wg, wu = (synth.make_weights(dtype, N, K, s) for s in (52, 53))
    x = synth.make_x(M, K, seed=M) * np.float32(1e-2)
    y = ops.ffn_up_fused(torch.from_numpy(x).cuda(), dev_weight(dtype, wg, N, K),
                         dev_weight(dtype, wu, N, K))
    g, u = (oracle.matmul_f64(dtype, x, w, N, K) for w in (wg, wu))
    assert_close_silu_mul(y.cpu().numpy(), g, u, x, wmax(dtype, [wg, wu], K), f"{dtype} {M}x{N}x{K}")


def test_q6k_four_tokens_on_many_rows():
    # as five tokens: the same kernel, a token's bits its own
    N, K = 24001, 2048
    W = dev_weight(F.Q6_K, synth.make_weights(F.Q6_K, N, K, 90), N, K)
    x = torch.from_numpy(synth.make_x(5, K, seed=91)).cuda()
    assert torch.equal(ops.matmul_transB(x[:4], W), ops.matmul_transB(x, W)[:4])


# Sizes on both sides of the line between this kernel and the band kernel, whose
# bands fill their rounds up to 16384 rows: one row more or less, other counts of tiles
@pytest.mark.parametrize("dtype", ALL)
@pytest.mark.parametrize("M,N,K", [(4, 12288, 4096), (8, 12289, 4096), (16, 16385, 2816), (5, 8200, 5632)])
def test_band_or_shared_operands(dtype, M, N, K):
    test_shapes(dtype, M, N, K)


@pytest.mark.parametrize("dtype", ALL)
@pytest.mark.parametrize("M,N,K", [(5, 1001, 256), (8, 6400, 2048), (16, 12289, 3584), (3, 16385, 1024)])
def test_pair_band_or_shared_operands(dtype, M, N, K):
    test_gate_up_pair(dtype, M, N, K)
