"""The tiled FP64 products (plane-fed and batched) carry RPL = 16 or 8 rows of
outputs per lane through DPP row broadcasts: every form bit for bit the
oracle's restatement at the edges of the 64- and 32-row tiles, of the k-slices
(8 and 16 k) and of the operands inside the batched tiles' buffer loads, with
padded leading dimensions (NaN on the inputs, a sentinel on the outputs), and
at leading dimensions beyond the buffer loads' 32-bit offsets."""
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

# one row / column / k past and short of a tile, a lane's rows and a slice
EDGES = [(63, 65, 17), (64, 64, 16), (65, 33, 15), (33, 129, 8), (31, 31, 7), (97, 1, 24), (17, 63, 33), (1, 65, 40)]


@pytest.mark.parametrize("rows", [64, 32])
@pytest.mark.parametrize("m,n,k", EDGES)
def test_plane_tiles_edges(ctx, rows, m, n, k):
    print("rows=%d m=%d n=%d k=%d" % (rows, m, n, k), flush=True)
    L = vcp_amd.lib()
    rng = np.random.default_rng(m * 7919 + n * 31 + k)
    lda, ldb, ldc = m + PAD, k + PAD, m + PAD
    IA = W.wide_exponent_intervals(rng, m, k, rad_exp=-20)
    IB = W.wide_exponent_intervals(rng, k, n, rad_exp=-20)
    A, B = _wide(rng, m, k), _wide(rng, k, n)
    dIA, dIB, dA, dB = _dev_iv(IA, lda), _dev_iv(IB, ldb), _dev_pt(A, lda), _dev_pt(B, ldb)
    ctx.set_param(vcp_amd.PARAM_PLANE_ROWS, rows)
    try:
        for fn, a, b, want in (("vcphip_igemm_ip_dev", dIA, dB, O.pidblas_mul_im_m(IA, B)),
                               ("vcphip_igemm_pi_dev", dA, dIB, O.pidblas_mul_m_im(A, IB))):
            C = _out_iv(m, n, ldc)
            _ok(getattr(L, fn)(ctx._h, m, n, k, a.data_ptr(), lda, b.data_ptr(), ldb, C.data_ptr(), ldc), fn)
            ctx.synchronize()
            assert np.array_equal(_read_iv(C, m), want), fn
        C = _out_iv(m, n, ldc)
        _ok(L.vcphip_igemm_dev(ctx._h, vcp_amd.FORM_PLAIN, m, n, k, dIA.data_ptr(), lda, dIB.data_ptr(), ldb,
                               C.data_ptr(), ldc), "igemm_dev")
        ctx.synchronize()
        assert np.array_equal(_read_iv(C, m), O.pidblas_mulmm(IA, IB))
        U, D = (torch.full((n, ldc), SENTINEL, dtype=torch.float64, device="cuda") for _ in range(2))
        torch.cuda.synchronize()
        _ok(L.vcphip_gemm_rurd_dev(ctx._h, m, n, k, dA.data_ptr(), lda, dB.data_ptr(), ldb, U.data_ptr(),
                                   D.data_ptr(), ldc, 0), "gemm_rurd_dev")
        ctx.synchronize()
        for t, sign in ((U, 1), (D, -1)):
            h = t.cpu().numpy()
            assert (h[:, m:] == SENTINEL).all() and np.array_equal(h[:, :m].T, O.rgemm(A, B, sign))
        # the same tiles of A^T A (k x n operand)
        C = _out_iv(n, n, n + PAD)
        _ok(L.vcphip_igemm_tn_dev(ctx._h, k, n, dIB.data_ptr(), ldb, C.data_ptr(), n + PAD), "igemm_tn_dev")
        ctx.synchronize()
        assert np.array_equal(_read_iv(C, n), O.pidblas_mulltmm(IB))
        C = _out_iv(n, n, n + PAD)
        _ok(L.vcphip_vgemm_tn_dev(ctx._h, k, n, dB.data_ptr(), ldb, C.data_ptr(), n + PAD), "vgemm_tn_dev")
        ctx.synchronize()
        assert np.array_equal(_read_iv(C, n), O.pidblas_vmulmm(B))
    finally:
        ctx.set_param(vcp_amd.PARAM_PLANE_ROWS, 0)


@pytest.mark.parametrize("tiles", [vcp_amd.BATCH_TILES_64, vcp_amd.BATCH_TILES_EDGE, vcp_amd.BATCH_TILES_32])
def test_batched_tiles_edges(ctx, tiles):
    L = vcp_amd.lib()
    rng = np.random.default_rng(tiles)
    probs = []
    for m, n, k in EDGES:
        IA = W.wide_exponent_intervals(rng, m, k, rad_exp=-20)
        IB = W.wide_exponent_intervals(rng, k, n, rad_exp=-20)
        probs.append((m, n, k, IA, IB, _dev_iv(IA, m + PAD), _dev_iv(IB, k + PAD), _out_iv(m, n, m + PAD)))
    ctx.set_param(vcp_amd.PARAM_BATCH_TILES, tiles)
    try:
        ctx.igemm_batched_dev([p[0] for p in probs], [p[1] for p in probs], [p[2] for p in probs],
                              [p[5].data_ptr() for p in probs], [p[0] + PAD for p in probs],
                              [p[6].data_ptr() for p in probs], [p[2] + PAD for p in probs],
                              [p[7].data_ptr() for p in probs], [p[0] + PAD for p in probs])
        ctx.synchronize()
        for m, n, k, IA, IB, _, _, C in probs:
            assert np.array_equal(_read_iv(C, m), O.pidblas_mulmm(IA, IB)), (m, n, k)
        ns = [1, 7, 31, 33, 64, 65, 97]
        Rs = [_wide(rng, n, n) for n in ns]
        As = [W.wide_exponent_intervals(rng, n, n, rad_exp=-20) for n in ns]
        dR, dA = [_dev_pt(R, n + PAD) for R, n in zip(Rs, ns)], [_dev_iv(A, n + PAD) for A, n in zip(As, ns)]
        Cs = [_out_iv(n, n, n + PAD) for n in ns]
        nub = torch.zeros(len(ns), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        ld = [n + PAD for n in ns]
        vcp_amd.residual_batched_dev(ctx, ns, [t.data_ptr() for t in dR], ld, [t.data_ptr() for t in dA], ld,
                                     [t.data_ptr() for t in Cs], ld, nub.data_ptr())
        ctx.synchronize()
        for n, R, A, C, g in zip(ns, Rs, As, Cs, nub.cpu().numpy()):
            Co, go = O.residual(R, A)
            assert np.array_equal(_read_iv(C, n), Co) and g == go, n
    finally:
        ctx.set_param(vcp_amd.PARAM_BATCH_TILES, 0)


def test_batched_tiles_large_leading_dimension(ctx):
    """a leading dimension of 2^21 rows takes the tiles' 64-bit addresses"""
    n, ld = 65, 1 << 21
    rng = np.random.default_rng(11)
    R, A = _wide(rng, n, n), W.wide_exponent_intervals(rng, n, n, rad_exp=-20)
    dR = torch.full((n, ld), float("nan"), dtype=torch.float64, device="cuda")
    dA = torch.full((n, ld, 2), float("nan"), dtype=torch.float64, device="cuda")
    dR[:, :n] = torch.from_numpy(np.ascontiguousarray(R.T)).cuda()
    dA[:, :n] = torch.from_numpy(np.ascontiguousarray(A.transpose(1, 0, 2))).cuda()
    C, nub = _out_iv(n, n, n), torch.zeros(1, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    vcp_amd.residual_batched_dev(ctx, [n], [dR.data_ptr()], [ld], [dA.data_ptr()], [ld], [C.data_ptr()], [n],
                                 nub.data_ptr())
    ctx.synchronize()
    Co, go = O.residual(R, A)
    assert np.array_equal(_read_iv(C, n), Co) and nub.item() == go
    C = _out_iv(n, n, n)
    ctx.igemm_batched_dev([n], [n], [n], [dA.data_ptr()], [ld], [dA.data_ptr()], [ld], [C.data_ptr()], [n])
    ctx.synchronize()
    assert np.array_equal(_read_iv(C, n), O.pidblas_mulmm(A, A))
