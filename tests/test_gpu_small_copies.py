"""Host-pointer products below 8 MiB go through one pinned buffer that grows and
is handed out in turn: operands of different sizes in a row, leading dimensions
above the row count, batched problems, changed streams.  Bit for bit the
device-pointer product, padding untouched."""
import numpy as np
import pytest
import torch

import oracle_ffi as O
import vcp_amd
from vcp_amd import workloads as W

pytestmark = pytest.mark.gpu


def _padded(rng, rows, cols, ld):
    X = O.pairs(ld, cols)
    X[...] = 7.0
    X[:rows] = W.wide_exponent_intervals(rng, rows, cols)
    return X


def _reference(ctx, A, B):
    m, n, k = A.shape[0], B.shape[1], A.shape[1]
    dA = torch.from_numpy(np.ascontiguousarray(A.transpose(1, 0, 2))).cuda()
    dB = torch.from_numpy(np.ascontiguousarray(B.transpose(1, 0, 2))).cuda()
    dC = torch.empty((n, m, 2), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    ctx.igemm_dev(vcp_amd.FORM_PLAIN, m, n, k, dA.data_ptr(), m, dB.data_ptr(), k, dC.data_ptr(), m)
    ctx.synchronize()
    return dC.cpu().numpy().transpose(1, 0, 2)


# (m, n, k): one element; a few kB; 1 MB blocks that outgrow the first buffer;
# just under and over 8 MiB per operand (724^2 and 725^2 x 16 B)
SIZES = [(1, 1, 1), (5, 3, 70), (96, 96, 96), (257, 200, 255), (5, 3, 70), (700, 64, 724), (724, 30, 724),
         (725, 30, 725), (64, 64, 64)]


def test_sizes_in_a_row_strided():
    ctx = vcp_amd.Context()
    L = vcp_amd.lib()
    rng = np.random.default_rng(5)
    streams = [torch.cuda.Stream() for _ in range(2)]
    for i, (m, n, k) in enumerate(SIZES):
        ctx.set_stream(streams[i % 2].cuda_stream if i % 3 else 0)
        lda, ldb, ldc = m + i % 2, k + 3 * (i % 2), m + 2 * (i % 2)
        A, B = _padded(rng, m, k, lda), _padded(rng, k, n, ldb)
        C = O.pairs(ldc, n)
        C[...] = 5.0
        assert L.vcphip_igemm(ctx._h, 0, m, n, k, A.ctypes.data, lda, B.ctypes.data, ldb, C.ctypes.data, ldc) == 0
        assert np.array_equal(C[:m], _reference(ctx, A[:m], B[:k])), (m, n, k)
        assert (C[m:] == 5.0).all()


def test_batched_pieces(ctx):
    rng = np.random.default_rng(6)
    sizes = [(1, 1, 1), (40, 33, 21), (64, 1, 100), (130, 90, 65), (3, 200, 17)]
    As = [W.wide_exponent_intervals(rng, m, k) for m, n, k in sizes]
    Bs = [W.wide_exponent_intervals(rng, k, n) for m, n, k in sizes]
    for A, B, C in zip(As, Bs, ctx.igemm_batched(As, Bs)):
        assert np.array_equal(C, _reference(ctx, A, B))
