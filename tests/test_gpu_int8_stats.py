"""Scales, norms and residue splits of both int8 operands, taken by one launch
each: bit-identical to the oracle at the edges of the row groups (8), column
groups (4 interval, 8 dd), 256-k norm chunks and pairs of chunks, and with
magnitudes that put the row maximum at the last k."""
import numpy as np
import pytest

import oracle_ffi as O
import vcp_amd
from vcp_amd import workloads as W

pytestmark = pytest.mark.gpu

SIZES = [(1, 5, 255), (7, 4, 256), (8, 3, 257), (9, 1, 511), (17, 9, 512), (3, 8, 513), (2, 2, 1023), (8, 4, 1025),
         (15, 7, 2049), (257, 130, 2), (1, 1, 64)]


def _last_k_largest(A, axis):
    idx = [slice(None)] * A.ndim
    idx[axis] = -1
    A[tuple(idx)] *= 2.0 ** 20
    return A


def _dd(rng, r, c):
    A = O.pairs(r, c)
    A[..., 0] = rng.standard_normal((r, c)) * np.exp2(rng.integers(-20, 21, (r, c)))
    A[..., 1] = A[..., 0] * 2.0 ** -54 * rng.uniform(-1, 1, (r, c))
    return A


@pytest.mark.parametrize("m,n,k", SIZES)
def test_interval_stats_edges(ctx, m, n, k):
    rng = np.random.default_rng(m + 31 * n + 101 * k)
    A = _last_k_largest(W.wide_exponent_intervals(rng, m, k), 1)
    B = _last_k_largest(W.wide_exponent_intervals(rng, k, n), 0)
    A[m // 2, :, :] = 0.0
    ctx.set_param(vcp_amd.PARAM_OZ_NMOD, 16)
    try:
        C = ctx.igemm(A, B, vcp_amd.FORM_OZAKI)
    finally:
        ctx.set_param(vcp_amd.PARAM_OZ_NMOD, 0)
    assert np.array_equal(C, O.ozaki_igemm(A, B, 16))


@pytest.mark.parametrize("m,n,k", SIZES)
def test_dd_stats_edges(ctx, m, n, k):
    rng = np.random.default_rng(m + 37 * n + 103 * k)
    nmod = O.dd_default_nmod(k)
    A, B = _last_k_largest(_dd(rng, m, k), 1), _last_k_largest(_dd(rng, k, n), 0)
    assert np.array_equal(ctx.ddgemm(A, B), O.ozaki_ddgemm(A, B, nmod))
    At = O.pairs(k, m)
    At[...] = A.transpose(1, 0, 2)
    assert np.array_equal(ctx.ddgemm_ta(At, B), O.ozaki_ddgemm(A, B, nmod))
    assert np.array_equal(ctx.ddgemm_tn(B), O.ozaki_ddgemm(B, None, nmod))
