"""The per-stream workspace of the M > 1 matrix-core path: reserved up front
it lets a call be captured into a HIP graph (every replay matches the eager
result); during capture a call that would have to grow it fails with
FQ_ERR_WORKSPACE instead of allocating."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from forge_amd import _lib, synth
from forge_amd import formats as F

pytestmark = pytest.mark.gpu


def _mm(L, dtype, x, w, y, M, K, N, stream):
    return L.fq_matmul_transB(dtype, x.data_ptr(), w.data_ptr(), None, 0, 0, y.data_ptr(), M, K,
                              N, stream)


def test_reserved_workspace_graph_replays():
    L = _lib.lib()
    dtype, M, K, N = F.Q4_K, 16, 4096, 2000  # MFMA path with K-splits
    w = torch.from_numpy(synth.make_weights(dtype, N, K, 31).reshape(-1)).cuda()
    x = torch.from_numpy(synth.make_x(M, K, 32)).cuda()
    side = torch.cuda.Stream()
    y_eager = torch.empty(M, N, device="cuda")
    y_graph = torch.empty(M, N, device="cuda")
    with torch.cuda.stream(side):
        assert L.fq_reserve_workspace(M, K, N, side.cuda_stream) == 0
        assert _mm(L, dtype, x, w, y_eager, M, K, N, side.cuda_stream) == 0
    torch.cuda.synchronize()
    ref = y_eager.cpu().numpy()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        st = _mm(L, dtype, x, w, y_graph, M, K, N, side.cuda_stream)
    assert st == 0
    for r in range(3):
        y_graph.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(y_graph.cpu().numpy(), ref, err_msg=f"replay {r}")
        # eager work on the same workspace between replays
        with torch.cuda.stream(side):
            assert _mm(L, dtype, x * 2, w, y_eager, M, K, N, side.cuda_stream) == 0
        torch.cuda.synchronize()
    del g
    assert L.fq_release_workspace(side.cuda_stream) == 0


def test_growth_under_capture_is_refused():
    L = _lib.lib()
    dtype, M, K, N = F.Q8_0, 24, 2048, 1024
    w = torch.from_numpy(synth.make_weights(dtype, N, K, 33).reshape(-1)).cuda()
    x = torch.from_numpy(synth.make_x(M, K, 34)).cuda()
    y = torch.empty(M, N, device="cuda")
    side = torch.cuda.Stream()  # a fresh stream: no workspace yet
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        st = _mm(L, dtype, x, w, y, M, K, N, side.cuda_stream)
    assert st == _lib.FQ_ERR_WORKSPACE
    assert b"fq_reserve_workspace" in L.fq_status_str(st)
    del g
    # outside capture the same call grows the workspace and runs
    with torch.cuda.stream(side):
        assert _mm(L, dtype, x, w, y, M, K, N, side.cuda_stream) == 0
    torch.cuda.synchronize()
    assert np.isfinite(y.cpu().numpy()).all()


@pytest.mark.parametrize("dtype,M,K,N", [(F.Q8_0, 40, 4096, 256), (F.Q4_0, 512, 1280, 4096),
                                         (F.Q4_K, 16, 4096, 2000), (F.Q8_0, 8, 2048, 3000),
                                         (F.Q6_K, 96, 2048, 1500), (F.Q4_K, 8, 18944, 3584),
                                         (F.Q6_K, 2, 18944, 3584), (F.Q4_0, 3, 18944, 3584),
                                         (F.Q6_K, 8, 18944, 3584), (F.Q8_0, 6, 18944, 3584),
                                         (F.Q4_1, 16, 4096, 1000), (F.Q5_K, 2, 18944, 3584)])
def test_reserve_then_capture_first(dtype, M, K, N):
    # fq_reserve_workspace alone (no eager call first) must cover the call's
    # kernel choice: the prefill kernel (Q8_0 / Q4_0, up to 16 K-splits; Q6_K
    # with its rewritten rows), the MMQ and small-batch paths (the band
    # kernel with K split over four slabs at 3584 x 18944, on Q4_K, Q4_0,
    # Q4_1, Q8_0 and Q6_K) and the batch-1 kernel over two or three tokens
    # with K split into slabs.  Three
    # replays, each checked against the eager call, with eager work between
    # them
    L = _lib.lib()
    w = torch.from_numpy(synth.make_weights(dtype, N, K, 41).reshape(-1)).cuda()
    x = torch.from_numpy(synth.make_x(M, K, 42)).cuda()
    y_graph = torch.empty(M, N, device="cuda")
    y_eager = torch.empty(M, N, device="cuda")
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    assert L.fq_reserve_workspace(M, K, N, side.cuda_stream) == 0
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        st = _mm(L, dtype, x, w, y_graph, M, K, N, side.cuda_stream)
    assert st == 0, L.fq_status_str(st)
    with torch.cuda.stream(side):
        assert _mm(L, dtype, x, w, y_eager, M, K, N, side.cuda_stream) == 0
    torch.cuda.synchronize()
    ref = y_eager.cpu().numpy()
    for _ in range(3):
        y_graph.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(y_graph.cpu().numpy(), ref)
        with torch.cuda.stream(side):
            assert _mm(L, dtype, x, w, y_eager, M, K, N, side.cuda_stream) == 0
        torch.cuda.synchronize()
    del g
    assert L.fq_release_workspace(side.cuda_stream) == 0


def test_fused_qkv_small_batch_graph_replays():
    # fused QKV at 8 tokens under capture after fq_reserve_workspace: the
    # band kernel's shared token operands need slot 0 at its largest band
    # size, which the reserve covers; every replay equals the eager call
    from forge_amd import ops
    L = _lib.lib()
    dtype, M, K, ns = F.Q4_K, 8, 4096, (4096, 1024, 1024)
    Ws = [ops.QWeight.from_numpy(synth.make_weights(dtype, n, K, 90 + i), dtype, n, K,
                                 device="cuda") for i, n in enumerate(ns)]
    x = torch.from_numpy(synth.make_x(M, K, 95)).cuda()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    assert L.fq_reserve_workspace(M, K, max(ns), side.cuda_stream) == 0
    with torch.cuda.stream(side):
        ref = ops.fused_qkv(x, *Ws).clone()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        y = ops.fused_qkv(x, *Ws)
    for _ in range(3):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ref)
        with torch.cuda.stream(side):
            ops.fused_qkv(x * 2, *Ws)
        torch.cuda.synchronize()
    del g
    assert L.fq_release_workspace(side.cuda_stream) == 0


def _fused(op, dtype, K, ns):
    """x -> a fused call over matrices of ns rows."""
    from forge_amd import ops
    Ws = [ops.QWeight.from_numpy(synth.make_weights(dtype, n, K, 110 + i), dtype, n, K, device="cuda")
          for i, n in enumerate(ns)]
    fn = ops.fused_qkv if op == "qkv" else ops.ffn_up_fused
    return lambda x: fn(x, *Ws)


# Fused launches after a reserve for larger sizes: smaller K and N can take more
# K-splits, three matrices more rows than any one.  The reserve covers them, so
# the captured call is the eager one and neither allocates: the shared-operand
# kernel (2..32 tokens) and the prefill kernels.
@pytest.mark.parametrize("op,dtype,M,K,ns,reserve", [
    ("pair", F.Q6_K, 307, 3584, (738, 738), (307, 4864, 739)),
    ("pair", F.Q6_K, 408, 4096, (365, 365), (408, 5632, 365)),
    ("qkv", F.Q8_0, 161, 4096, (470, 470, 470), (161, 4096, 470)),
    ("pair", F.Q6_K, 15, 11520, (764, 764), (15, 12288, 764)),
    ("pair", F.Q4_0, 3, 4096, (5632, 5632), (4, 4096, 5632)),
    ("qkv", F.Q5_1, 27, 2048, (2048, 256, 256), (32, 5632, 2048)),
    ("pair", F.Q5_K, 77, 4096, (14336, 14336), (77, 14336, 14336))])
def test_reserve_covers_fused_launches(op, dtype, M, K, ns, reserve):
    L = _lib.lib()
    run = _fused(op, dtype, K, ns)
    x = torch.from_numpy(synth.make_x(M, K, 121) * np.float32(1e-2)).cuda()
    ref = run(x)  # on a workspace of its own that grows as it likes
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    assert L.fq_reserve_workspace(*reserve, side.cuda_stream) == 0
    with torch.cuda.stream(side):
        torch.empty_like(ref)  # the result's memory, before free memory is read
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        y = run(x)
    for _ in range(3):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ref)
        with torch.cuda.stream(side):
            assert torch.equal(run(x), ref)
            run(x * 2)
        torch.cuda.synchronize()
    grown = free - torch.cuda.mem_get_info()[0]
    assert grown < 32 << 20, f"{grown} bytes allocated after the reserve"  # torch's own blocks
    del g
    assert L.fq_release_workspace(side.cuda_stream) == 0


def test_reserve_is_no_larger_than_its_calls_need():
    # 512 tokens at 14336: the operands (33 MB), the rewritten rows of one Q6_K
    # matrix (231 MB), at most 256 MiB of slabs, the rows of a fused op (59 MB)
    L = _lib.lib()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    assert L.fq_reserve_workspace(512, 14336, 14336, side.cuda_stream) == 0
    assert free - torch.cuda.mem_get_info()[0] <= 600 << 20
    assert L.fq_release_workspace(side.cuda_stream) == 0


# No reserve, the workspace sized by an eager call of more tokens: a plan for
# fewer tokens can want more of it (parts of row tiles, K-splits), so under
# capture it makes do with what is there
@pytest.mark.parametrize("op,dtype,Mw,M,K,ns", [
    ("one", F.Q4_K, 32, 17, 1024, (8192,)), ("one", F.Q4_K, 32, 19, 4096, (4096,)),
    ("pair", F.Q4_K, 32, 17, 4096, (14336, 14336)), ("qkv", F.Q4_K, 32, 19, 4096, (2048, 512, 512)),
    ("pair", F.Q8_0, 256, 130, 4096, (2048, 2048)), ("one", F.Q5_K, 512, 130, 4096, (4096,))])
def test_capture_of_fewer_tokens_than_warmed_up(op, dtype, Mw, M, K, ns):
    from forge_amd import ops
    L = _lib.lib()
    if op == "one":
        W = ops.QWeight.from_numpy(synth.make_weights(dtype, ns[0], K, 130), dtype, ns[0], K, device="cuda")
        run = lambda x: ops.matmul_transB(x, W)  # noqa: E731
    else:
        run = _fused(op, dtype, K, ns)
    x = torch.from_numpy(synth.make_x(Mw, K, 131) * np.float32(1e-2)).cuda()
    ref = run(x[:M])
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        run(x)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        y = run(x[:M])
    for _ in range(3):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert float((y - ref).norm() / ref.norm()) < 1e-6
        with torch.cuda.stream(side):
            assert torch.equal(run(x[:M]), ref)  # outside of capture it grows
        torch.cuda.synchronize()
    del g
    assert L.fq_release_workspace(side.cuda_stream) == 0


# Calls whose kernel an estimate chooses (band or shared operands), first
# under capture on a workspace that a call of other tokens sized: where the chosen
# one does not fit, another runs.  Each within 1e-6 of the exact result.
@pytest.mark.parametrize("op,dtype,Mw,M,K,ns", [
    ("pair", F.Q4_0, 2, 8, 2048, (6400, 6400)), ("pair", F.Q6_K, 2, 5, 256, (4096, 4096)),
    ("pair", F.Q5_0, 2, 8, 3584, (9472, 9472)), ("one", F.Q4_K, 17, 4, 4096, (11008,)),
    ("one", F.Q4_0, 17, 8, 5632, (12288,)), ("one", F.Q5_0, 17, 4, 4096, (12288,))])
def test_capture_where_estimates_choose(op, dtype, Mw, M, K, ns):
    from forge_amd import ops
    L = _lib.lib()
    if op == "one":
        W = ops.QWeight.from_numpy(synth.make_weights(dtype, ns[0], K, 140), dtype, ns[0], K, device="cuda")
        run = lambda x: ops.matmul_transB(x, W)  # noqa: E731
    else:
        run = _fused(op, dtype, K, ns)
    x = torch.from_numpy(synth.make_x(max(Mw, M), K, 141) * np.float32(1e-2)).cuda()
    ref = run(x[:M])
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        run(x[:Mw])
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        y = run(x[:M])
    for _ in range(3):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert float((y - ref).norm() / ref.norm()) < 2e-6
        with torch.cuda.stream(side):
            assert torch.equal(run(x[:M]), ref)
        torch.cuda.synchronize()
    del g
    assert L.fq_release_workspace(side.cuda_stream) == 0
