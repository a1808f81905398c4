"""The RU / RD point product moves its results, and the values it continues
from, between memory and the tile's lanes through LDS: bit for bit the oracle's
chains at the edges of the moved blocks (16 or 32 rows x 32 columns of a wave,
passes of 8, 16 or 32 columns), both tile heights, from zero and accumulating,
with padded leading dimensions whose padding stays as it was."""
import numpy as np
import pytest
import torch

import oracle_ffi as O
import vcp_amd
from test_gpu_planes import PAD, SENTINEL, _dev_pt, _ok, _wide, plane_rows  # noqa: F401

pytestmark = pytest.mark.gpu

SHAPES = [(1, 33, 5), (15, 1, 16), (16, 32, 17), (17, 65, 3), (31, 72, 16), (33, 40, 40), (63, 96, 8), (97, 31, 24),
          (128, 128, 1), (200, 201, 33)]


@pytest.mark.parametrize("acc", [0, 1])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_point_blocks_bitexact(ctx, plane_rows, m, n, k, acc):  # noqa: F811
    print("point blocks rows=%d m=%d n=%d k=%d acc=%d" % (plane_rows, m, n, k, acc), flush=True)
    rng = np.random.default_rng(m * 7919 + n * 31 + k)
    lda, ldb, ldc = m + PAD, k + PAD, m + PAD
    A, B = _wide(rng, m, k), _wide(rng, k, n)
    U0, D0 = _wide(rng, m, n), _wide(rng, m, n)
    dA, dB, dU, dD = _dev_pt(A, lda), _dev_pt(B, ldb), _dev_pt(U0, ldc), _dev_pt(D0, ldc)
    dU[:, m:] = SENTINEL
    dD[:, m:] = SENTINEL
    torch.cuda.synchronize()
    _ok(vcp_amd.lib().vcphip_gemm_rurd_dev(ctx._h, m, n, k, dA.data_ptr(), lda, dB.data_ptr(), ldb, dU.data_ptr(),
                                           dD.data_ptr(), ldc, acc), "gemm_rurd_dev")
    ctx.synchronize()
    for got, start, sign in ((dU, U0, 1), (dD, D0, -1)):
        g = got.cpu().numpy()
        assert (g[:, m:] == SENTINEL).all()
        want = O.rgemm(A, B, sign, C=np.asfortranarray(start.copy()), accumulate=bool(acc))
        assert np.array_equal(g[:, :m].T, want)
