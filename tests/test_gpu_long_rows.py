"""Row statistics of few long rows, split over workgroups along k (steps of 512)
and merged: bit for bit the oracle at the edges of the rule (k = 2560 is not
split, 2561 is; 2048 rows, 2049), with the row maximum at the last k, a zero row
and rows that are non-finite in the first and in the last part."""
import numpy as np
import pytest

import oracle_ffi as O
import vcp_amd
from vcp_amd import workloads as W

pytestmark = pytest.mark.gpu

SIZES = [(5, 2, 2560), (5, 3, 2561), (8, 1, 3072), (9, 2, 3073), (33, 1, 5000), (100, 2, 12289), (2048, 1, 2600),
         (2049, 1, 2600), (1, 1, 40000)]


def _mark(A, k):
    m = A.shape[0]
    A[:, -1] *= 2.0 ** 20
    if m >= 5:
        A[m // 2] = 0.0
        A[0, 3, 1] = np.inf
        A[1, k - 2, 0] = np.nan
        A[m - 1, k - 1, 0] = -np.inf
    return A


@pytest.mark.parametrize("m,n,k", SIZES)
def test_interval_long_rows(ctx, m, n, k):
    print("long rows m=%d n=%d k=%d" % (m, n, k), flush=True)
    rng = np.random.default_rng(m + 31 * n + 101 * k)
    A, B = _mark(W.wide_exponent_intervals(rng, m, k), k), W.wide_exponent_intervals(rng, k, n)
    ctx.set_param(vcp_amd.PARAM_OZ_NMOD, 16)
    ctx.set_param(vcp_amd.PARAM_OZ_RADIUS, vcp_amd.OZ_RADIUS_FULL)
    try:
        C = ctx.igemm(A, B, vcp_amd.FORM_OZAKI)
    finally:
        ctx.set_param(vcp_amd.PARAM_OZ_NMOD, 0)
        ctx.set_param(vcp_amd.PARAM_OZ_RADIUS, 0)
    assert np.array_equal(C, O.ozaki_igemm(A, B, 16, vcp_amd.OZ_RADIUS_FULL), equal_nan=True)


@pytest.mark.parametrize("m,n,k", SIZES)
def test_dd_long_rows(ctx, m, n, k):
    print("dd long rows m=%d n=%d k=%d" % (m, n, k), flush=True)
    rng = np.random.default_rng(m + 37 * n + 103 * k)
    A, B = _mark(W.dd_matrix(rng, m, k), k), W.dd_matrix(rng, k, n)
    assert np.array_equal(ctx.ddgemm(A, B), O.ozaki_ddgemm(A, B, O.dd_default_nmod(k)), equal_nan=True)
