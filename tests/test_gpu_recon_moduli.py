"""Reconstruction with one wave per 16 x 16 block (outputs of more than 8192
blocks) at every moduli count: the bits of the products of its row and column
halves, which take four waves per block and are compared with the oracle
elsewhere (a row's and a column's scales do not depend on the others)."""
import numpy as np
import pytest

import oracle_ffi as O
import vcp_amd
from vcp_amd import workloads as W
from test_gpu_recon_blocks import _dd

pytestmark = pytest.mark.gpu

M, N, K = 1449, 1467, 9   # 96 x 96 blocks once padded; 64 x 64 a half
RADII = [vcp_amd.OZ_RADIUS_FULL, vcp_amd.OZ_RADIUS_FOLDED, vcp_amd.OZ_RADIUS_HALF, vcp_amd.OZ_RADIUS_CEIL]


def _halves(product, A, B, C):
    for i in (slice(0, 1000), slice(1000, M)):
        for j in (slice(0, 1000), slice(1000, N)):
            assert np.array_equal(product(vcp_amd.as_pairs(A[i]), vcp_amd.as_pairs(B[:, j])), C[i, j])


@pytest.mark.parametrize("nmod", range(8, 21))
def test_interval_moduli(ctx, nmod):
    print("recon moduli", nmod, flush=True)
    rng = np.random.default_rng(nmod)
    A, B = W.wide_exponent_intervals(rng, M, K), W.wide_exponent_intervals(rng, K, N)
    A[M // 2] = 0.0
    B[:, N - 1] = 0.0
    ctx.set_param(vcp_amd.PARAM_OZ_NMOD, nmod)
    ctx.set_param(vcp_amd.PARAM_OZ_RADIUS, RADII[nmod % 4])
    try:
        _halves(lambda a, b: ctx.igemm(a, b, vcp_amd.FORM_OZAKI), A, B, ctx.igemm(A, B, vcp_amd.FORM_OZAKI))
        few = ctx.igemm(vcp_amd.as_pairs(A[:40]), vcp_amd.as_pairs(B[:, :50]), vcp_amd.FORM_OZAKI)
    finally:
        ctx.set_param(vcp_amd.PARAM_OZ_NMOD, 0)
        ctx.set_param(vcp_amd.PARAM_OZ_RADIUS, 0)
    assert np.array_equal(few, O.ozaki_igemm(vcp_amd.as_pairs(A[:40]), vcp_amd.as_pairs(B[:, :50]), nmod, RADII[nmod % 4]))


@pytest.mark.parametrize("nmod", range(24, 33))
def test_dd_moduli(ctx, nmod):
    print("recon dd moduli", nmod, flush=True)
    rng = np.random.default_rng(nmod)
    A, B = _dd(rng, M, K), _dd(rng, K, N)
    A[M // 2] = 0.0
    ctx.set_param(vcp_amd.PARAM_DD_NMOD, nmod)
    try:
        _halves(ctx.ddgemm, A, B, ctx.ddgemm(A, B))
        few = ctx.ddgemm(vcp_amd.as_pairs(A[:40]), vcp_amd.as_pairs(B[:, :50]))
    finally:
        ctx.set_param(vcp_amd.PARAM_DD_NMOD, 0)
    assert np.array_equal(few, O.ozaki_ddgemm(vcp_amd.as_pairs(A[:40]), vcp_amd.as_pairs(B[:, :50]), nmod))
