"""Products of k = 0 on device pointers: zeros with the signs of empty round-up
and round-down chains (intervals {-0, +0}, RU +0, RD -0), padding untouched,
operands never read; accumulating leaves the results as they are."""
import numpy as np
import pytest
import torch

import vcp_amd
from test_gpu_planes import PAD, SENTINEL, _ok

pytestmark = pytest.mark.gpu


def _same_bits(t, value):
    return bool((t.view(torch.int64) == int(np.float64(value).view(np.int64))).all())


@pytest.mark.parametrize("m,n", [(1, 1), (255, 3), (257, 2), (5, 70000)])
def test_empty_products(ctx, m, n):
    L, ld = vcp_amd.lib(), m + PAD
    out = lambda e: torch.full((n, ld, e), SENTINEL, dtype=torch.float64, device="cuda")  # noqa: E731
    nul = torch.zeros(1, dtype=torch.float64, device="cuda").data_ptr()   # one element: nothing of it may be used
    for call in (lambda C: L.vcphip_igemm_dev(ctx._h, vcp_amd.FORM_PLAIN, m, n, 0, nul, m, nul, 1, C, ld),
                 lambda C: L.vcphip_igemm_ip_dev(ctx._h, m, n, 0, nul, m, nul, 1, C, ld),
                 lambda C: L.vcphip_igemm_pi_dev(ctx._h, m, n, 0, nul, m, nul, 1, C, ld)):
        C = out(2)
        torch.cuda.synchronize()
        _ok(call(C.data_ptr()), "product")
        ctx.synchronize()
        assert _same_bits(C[:, :m, 0].contiguous(), -0.0) and _same_bits(C[:, :m, 1].contiguous(), 0.0)
        assert (C[:, m:] == SENTINEL).all()
    for acc in (0, 1):
        U, D = out(1), out(1)
        torch.cuda.synchronize()
        _ok(L.vcphip_gemm_rurd_dev(ctx._h, m, n, 0, nul, m, nul, 1, U.data_ptr(), D.data_ptr(), ld, acc), "rurd")
        ctx.synchronize()
        assert _same_bits(U[:, :m].contiguous(), SENTINEL if acc else 0.0)
        assert _same_bits(D[:, :m].contiguous(), SENTINEL if acc else -0.0)
        assert (U[:, m:] == SENTINEL).all() and (D[:, m:] == SENTINEL).all()


@pytest.mark.parametrize("n", [1, 65, 300])
def test_empty_gram_matrices(ctx, n):
    L, ld = vcp_amd.lib(), n + PAD
    nul = torch.zeros(1, dtype=torch.float64, device="cuda").data_ptr()
    for f in (L.vcphip_igemm_tn_dev, L.vcphip_vgemm_tn_dev):
        C = torch.full((n, ld, 2), SENTINEL, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        _ok(f(ctx._h, 0, n, nul, 1, C.data_ptr(), ld), "tn")
        ctx.synchronize()
        assert _same_bits(C[:, :n, 0].contiguous(), -0.0) and _same_bits(C[:, :n, 1].contiguous(), 0.0)
        assert (C[:, n:] == SENTINEL).all()
