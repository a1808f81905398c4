"""The row-serial products (few columns, or too small for tiles): every form
bit for bit the oracle's restatement at the edges of the kernel's blocks (8
rows; 8, 16, 32 and 64 columns; stages of 96, 64 and 32 k, zero terms up to a
multiple of 16), with padded leading dimensions whose padding is NaN on the
inputs and a sentinel on the outputs; and the verified solve's steps built on
the same kernel at the numbers of right-hand sides where its shape or route
changes."""
import numpy as np
import pytest
import torch

import oracle_ffi as O
import vcp_amd
from vcp_amd import workloads as W
from test_gpu_planes import PAD, SENTINEL, _dev_iv, _dev_pt, _ok, _read_iv, _wide
from test_gpu_planes import _out_iv as _out_async

pytestmark = pytest.mark.gpu


def _out_iv(rows, cols, ld):
    t = _out_async(rows, cols, ld)
    torch.cuda.synchronize()   # the fill runs on torch's stream, the product on the context's
    return t

# columns per workgroup: 8 up to n = 8 and for small grids, 16 up to n = 16,
# 32 at (640, 64), 64 at (1200, 17) and (1201, 65)
SHAPES = [(1, 1, 1), (7, 8, 15), (8, 9, 16), (9, 16, 17), (23, 17, 96), (16, 1, 97), (40, 33, 64), (15, 65, 65),
          (640, 64, 33), (1200, 17, 40), (1201, 65, 31), (300, 2, 700), (3, 700, 193)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_thin_products_bitexact(ctx, m, n, k):
    print("thin m=%d n=%d k=%d" % (m, n, k), flush=True)
    L = vcp_amd.lib()
    rng = np.random.default_rng(m * 7919 + n * 31 + k)
    lda, ldb, ldc = m + PAD, k + PAD, m + PAD
    IA = W.wide_exponent_intervals(rng, m, k, rad_exp=-20)
    IB = W.wide_exponent_intervals(rng, k, n, rad_exp=-20)
    A, B = _wide(rng, m, k), _wide(rng, k, n)
    dIA, dIB, dA, dB = _dev_iv(IA, lda), _dev_iv(IB, ldb), _dev_pt(A, lda), _dev_pt(B, ldb)
    C = _out_iv(m, n, ldc)
    _ok(L.vcphip_igemm_dev(ctx._h, vcp_amd.FORM_PLAIN, m, n, k, dIA.data_ptr(), lda, dIB.data_ptr(), ldb,
                           C.data_ptr(), ldc), "igemm_dev")
    ctx.synchronize()
    assert np.array_equal(_read_iv(C, m), O.pidblas_mulmm(IA, IB))
    C = _out_iv(m, n, ldc)
    _ok(L.vcphip_igemm_ip_dev(ctx._h, m, n, k, dIA.data_ptr(), lda, dB.data_ptr(), ldb, C.data_ptr(), ldc), "ip")
    ctx.synchronize()
    assert np.array_equal(_read_iv(C, m), O.pidblas_mul_im_m(IA, B))
    C = _out_iv(m, n, ldc)
    _ok(L.vcphip_igemm_pi_dev(ctx._h, m, n, k, dA.data_ptr(), lda, dIB.data_ptr(), ldb, C.data_ptr(), ldc), "pi")
    ctx.synchronize()
    assert np.array_equal(_read_iv(C, m), O.pidblas_mul_m_im(A, IB))
    for acc in (0, 1):   # point RU / RD, from zero and onto existing values
        U0, D0 = _wide(rng, m, n), _wide(rng, m, n)
        dU, dD = _dev_pt(U0, ldc), _dev_pt(D0, ldc)
        dU[:, m:] = SENTINEL
        dD[:, m:] = SENTINEL
        torch.cuda.synchronize()
        _ok(L.vcphip_gemm_rurd_dev(ctx._h, m, n, k, dA.data_ptr(), lda, dB.data_ptr(), ldb, dU.data_ptr(),
                                   dD.data_ptr(), ldc, acc), "gemm_rurd_dev")
        ctx.synchronize()
        u, d = dU.cpu().numpy(), dD.cpu().numpy()
        assert (u[:, m:] == SENTINEL).all() and (d[:, m:] == SENTINEL).all()
        for got, start, sign in ((u, U0, 1), (d, D0, -1)):
            assert np.array_equal(got[:, :m].T,
                                  O.rgemm(A, B, sign, C=np.asfortranarray(start.copy()), accumulate=bool(acc)))


@pytest.mark.parametrize("special", [np.inf, -np.inf, np.nan])
def test_thin_products_nonfinite(ctx, special):
    """a non-finite end meets the same chains as in the tiles, padding included"""
    rng = np.random.default_rng(5)
    IA, IB = W.uniform_intervals(rng, 11, 19, -20), W.uniform_intervals(rng, 19, 3, -20)
    IA[4, 18, 1] = special
    IB[2, 1, 0] = special
    C = ctx.igemm(IA, IB)
    assert np.array_equal(C, O.pidblas_mulmm(IA, IB), equal_nan=True)


@pytest.mark.parametrize("n,nrhs,rows", [(40, 8, 0), (41, 9, 0), (95, 65, 0), (97, 40, 32), (200, 1, 0)])
def test_lss_right_hand_sides(ctx, n, nrhs, rows):
    """8 right-hand sides per workgroup, 64 above 8, and (rows: a forced plane
    height) the tiled route of many right-hand sides; the batched form agrees"""
    rng = np.random.default_rng(n * 100 + nrhs)
    A = rng.uniform(-1, 1, (n, n)) + 0.5 * n * np.eye(n)
    b = rng.uniform(-1, 1, (n, nrhs))
    IA = W.interval_from_midrad(A, np.ldexp(np.abs(A), -30))
    Ib = W.interval_from_midrad(b, np.ldexp(np.abs(b), -30))
    R = np.asfortranarray(np.linalg.inv(A))
    Xo, go, ok = O.lss(IA, Ib, R)
    assert ok
    ctx.set_param(vcp_amd.PARAM_PLANE_ROWS, rows)
    try:
        X, g = ctx.lss(IA, Ib, R)
    finally:
        ctx.set_param(vcp_amd.PARAM_PLANE_ROWS, 0)
    assert g == go and np.array_equal(X, Xo)
    I1 = vcp_amd.as_pairs(Ib[:, :1])
    Xb, gb = ctx.lss_batched([IA, IA], [Ib, I1], [R, R])
    assert gb[0] == go and np.array_equal(Xb[0], Xo)
    assert np.array_equal(Xb[1], O.lss(IA, I1, R)[0])
