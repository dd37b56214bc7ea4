"""The dequant kernel's chunks of 256 elements: rows that end inside a chunk,
a quad or a block, rows and outputs that are not whole 16-byte pieces."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from forge_amd import _lib, synth
from forge_amd import formats as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", sorted(F.FORMATS))
@pytest.mark.parametrize("N,K,shift", [(1, 1, 0), (5, 31, 0), (9, 256, 1), (33, 258, 0),
                                       (70, 1023, 0), (3, 1028, 2), (2049, 320, 0)])
def test_dequant_ragged_rows_and_bases(dtype, N, K, shift):
    be = F.fmt(dtype).block_elems
    w = synth.make_weights(dtype, N, -(-K // be) * be, seed=N + K)
    ref = oracle.dequant(dtype, w, N, K).reshape(N, K)
    # the weights 2 bytes and the result 4 * shift bytes past an aligned base
    wd = torch.zeros(w.size + 2, dtype=torch.uint8, device="cuda")
    wd[2:] = torch.from_numpy(w.reshape(-1)).cuda()
    out = torch.full((N * K + 8,), float("nan"), device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    assert _lib.lib().fq_dequant_rows(dtype, wd.data_ptr() + 2, out.data_ptr() + 4 * shift, N, K,
                                      st) == 0
    got = out.cpu().numpy()
    assert np.array_equal(got[shift:shift + N * K].view(np.uint32), ref.reshape(-1).view(np.uint32))
    assert np.isnan(got[:shift]).all() and np.isnan(got[shift + N * K:]).all()


# the longest row: its last chunk ends 31 below the largest int
def test_dequant_longest_row():
    K = 2 ** 31 - 32
    w = torch.randint(0, 256, (K // 32 * 18,), dtype=torch.uint8, device="cuda")
    w[0::18] = 0  # scales of 2^-14 and below
    w[1::18] &= 0x83
    out = torch.full((K,), float("nan"), device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    assert _lib.lib().fq_dequant_rows(F.Q4_0, w.data_ptr(), out.data_ptr(), 1, K, st) == 0
    assert not torch.isnan(out.sum())
    n = 4096  # of either end
    for s, o in ((w[:n // 32 * 18], out[:n]), (w[-n // 32 * 18:], out[-n:])):
        ref = oracle.dequant(F.Q4_0, s.cpu().numpy().reshape(1, -1), 1, n).reshape(n)
        assert np.array_equal(o.cpu().numpy().view(np.uint32), ref.view(np.uint32))
    assert _lib.lib().fq_dequant_rows(F.Q8_0, w.data_ptr(), out.data_ptr(), 1, K, st) == _lib.FQ_ERR_SHAPE
