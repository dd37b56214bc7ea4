"""Several matrices in one prefill launch (M > 32): tiles that do not span two
matrices, gate and up rows in one tile, with and without K-splits, against
the exact products; and the one-call-per-matrix path where the launch cannot
run (an unaligned matrix, a workspace that cannot grow under capture)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from forge_amd import _lib, ops, synth
from forge_amd import formats as F
from helpers import assert_close, assert_close_silu_mul
from test_gpu_parity import dev_weight

pytestmark = pytest.mark.gpu
PREFILL = [F.Q4_0, F.Q4_1, F.Q8_0, F.Q5_0, F.Q5_1, F.Q4_K, F.Q5_K, F.Q6_K]


def exact(dtype, x, w, K):
    return oracle.matmul_f64(dtype, x, w, w.shape[0], K)


def wmax(dtype, ws, K):
    return max(float(np.max(np.abs(oracle.dequant(dtype, w, w.shape[0], K)))) for w in ws)


@pytest.mark.parametrize("dtype", PREFILL)
@pytest.mark.parametrize("M,K,ns", [(33, 256, (257, 64, 1)), (130, 2048, (1, 300, 255)),
                                    (64, 512, (0, 96, 33)), (40, 768, (31, 0, 256))])
def test_qkv_one_launch(dtype, M, K, ns):
    ws = [synth.make_weights(dtype, n, K, 40 + i) for i, n in enumerate(ns)]
    x = synth.make_x(M, K, seed=M)
    W = [dev_weight(dtype, w, n, K) for w, n in zip(ws, ns)]
    y = ops.fused_qkv(torch.from_numpy(x).cuda(), *W)
    ref = np.concatenate([exact(dtype, x, w, K) for w in ws if w.shape[0]], axis=1)
    assert_close(y.cpu().numpy(), ref, x, np.array([wmax(dtype, [w for w in ws if len(w)], K)]),
                 f"qkv {dtype} {ns}")


@pytest.mark.parametrize("dtype", PREFILL)
@pytest.mark.parametrize("M,N,K", [(33, 1, 256), (64, 127, 512), (130, 129, 768), (96, 300, 2048)])
def test_gate_up_one_launch(dtype, M, N, K):
    wg, wu = (synth.make_weights(dtype, N, K, s) for s in (50, 51))
    x = synth.make_x(M, K, seed=M) * np.float32(1e-2)
    y = ops.ffn_up_fused(torch.from_numpy(x).cuda(), dev_weight(dtype, wg, N, K),
                         dev_weight(dtype, wu, N, K))
    assert_close_silu_mul(y.cpu().numpy(), exact(dtype, x, wg, K), exact(dtype, x, wu, K), x,
                          wmax(dtype, [wg, wu], K), f"gate/up {dtype} {M}x{N}x{K}")


def offset_weight(dtype, w, N, K, off):
    t = torch.zeros(w.size + off, dtype=torch.uint8, device="cuda")
    t[off:] = torch.from_numpy(w.reshape(-1)).cuda()
    return ops.QWeight(t[off:], dtype, N, K)


@pytest.mark.parametrize("dtype", [F.Q4_K, F.Q6_K, F.Q8_0])
def test_one_matrix_at_an_offset_base(dtype):
    M, N, K = 48, 200, 1024
    wg, wu = (synth.make_weights(dtype, N, K, s) for s in (60, 61))
    x = synth.make_x(M, K, seed=62) * np.float32(1e-2)
    xd = torch.from_numpy(x).cuda()
    G, U = dev_weight(dtype, wg, N, K), offset_weight(dtype, wu, N, K, 2)
    g, u = exact(dtype, x, wg, K), exact(dtype, x, wu, K)
    wm = wmax(dtype, [wg, wu], K)
    assert_close_silu_mul(ops.ffn_up_fused(xd, G, U).cpu().numpy(), g, u, x, wm, "gate/up offset")
    assert_close(ops.fused_qkv(xd, U, G, U).cpu().numpy(), np.concatenate([u, g, u], axis=1), x,
                 np.array([wm]), "qkv offset")


def test_capture_with_a_workspace_for_single_matrices():
    # the one-launch QKV wants a larger workspace than its matrices one by
    # one (16 K-splits of 3072 columns, the rewritten rows of three matrices);
    # where a reservation for smaller matrices cannot grow to it (capture) the
    # call still runs, one matrix at a time
    L = _lib.lib()
    dtype, M, K, ns = F.Q6_K, 64, 4096, (1024, 1024, 1024)
    ws = [torch.from_numpy(synth.make_weights(dtype, n, K, 70 + i).reshape(-1)).cuda()
          for i, n in enumerate(ns)]
    x = torch.from_numpy(synth.make_x(M, K, 73)).cuda()
    side = torch.cuda.Stream()
    y, ref = (torch.empty(M, sum(ns), device="cuda") for _ in range(2))

    def call(out):
        return L.fq_fused_qkv(dtype, x.data_ptr(), *(w.data_ptr() for w in ws), out.data_ptr(), M, K,
                              *ns, side.cuda_stream)

    with torch.cuda.stream(side):
        assert L.fq_reserve_workspace(M, K, 512, side.cuda_stream) == 0
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        st = call(y)
    assert st == 0
    with torch.cuda.stream(side):
        assert call(ref) == 0
    torch.cuda.synchronize()
    for _ in range(3):
        y.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert float((y - ref).norm() / ref.norm()) < 1e-6
        with torch.cuda.stream(side):
            assert call(ref) == 0
        torch.cuda.synchronize()
    del g
    assert L.fq_release_workspace(side.cuda_stream) == 0


def test_q6k_pair_beyond_the_rewrite_limit():
    # 167 MiB of rewritten rows: one call per matrix
    dtype, M, N, K = F.Q6_K, 33, 19000, 4096
    G, U = (dev_weight(dtype, synth.make_weights(dtype, N, K, s), N, K) for s in (80, 81))
    x = torch.from_numpy(synth.make_x(M, K, seed=82) * np.float32(1e-2)).cuda()
    ref = torch.nn.functional.silu(ops.matmul_transB(x, G)) * ops.matmul_transB(x, U)
    torch.testing.assert_close(ops.ffn_up_fused(x, G, U), ref, rtol=2e-6, atol=1e-9)
