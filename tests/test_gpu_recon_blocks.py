"""Reconstruction with one wave per 16 x 16 block (large outputs) and with four
(small ones), on both sides of the line and with ragged last blocks: the oracle's
bits, the padding between m and ldc untouched."""
import numpy as np
import pytest
import torch

import oracle_ffi as O
import vcp_amd
from vcp_amd import workloads as W

pytestmark = pytest.mark.gpu

# blocks of 16 x 16 over the padded output: 8 x 1024 = 8192 is the line
SIZES = [(113, 16300, 9), (113, 16401, 9), (1, 17, 5), (130, 8300, 7)]


def _dd(rng, r, c):
    A = O.pairs(r, c)
    A[..., 0] = rng.standard_normal((r, c)) * np.exp2(rng.integers(-30, 31, (r, c)))
    A[..., 1] = A[..., 0] * 2.0 ** -54 * rng.uniform(-1, 1, (r, c))
    return A


def _dev(X):
    return torch.from_numpy(np.ascontiguousarray(X.transpose(1, 0, 2))).cuda()


@pytest.mark.parametrize("form", ["interval", "dd"])
@pytest.mark.parametrize("m,n,k", SIZES)
def test_recon_blocks(ctx, m, n, k, form):
    rng = np.random.default_rng(m + 3 * n + 5 * k)
    make = _dd if form == "dd" else W.wide_exponent_intervals
    A, B = make(rng, m, k), make(rng, k, n)
    A[m // 2] = 0.0
    B[:, n - 1] = 0.0
    ldc = m + 3
    dA, dB = _dev(A), _dev(B)
    dC = torch.full((n, ldc, 2), 7.0, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    if form == "dd":
        assert vcp_amd.lib().vcphip_ddgemm_dev(ctx._h, m, n, k, dA.data_ptr(), m, dB.data_ptr(), k, dC.data_ptr(), ldc) == 0
        want = O.ozaki_ddgemm(A, B, O.dd_default_nmod(k))
    else:
        ctx.set_param(vcp_amd.PARAM_OZ_NMOD, 16)
        try:
            ctx.igemm_dev(vcp_amd.FORM_OZAKI, m, n, k, dA.data_ptr(), m, dB.data_ptr(), k, dC.data_ptr(), ldc)
        finally:
            ctx.set_param(vcp_amd.PARAM_OZ_NMOD, 0)
        want = O.ozaki_igemm(A, B, 16)
    ctx.synchronize()
    C = dC.cpu().numpy().transpose(1, 0, 2)
    assert np.array_equal(C[:m], want)
    assert (C[m:] == 7.0).all()
