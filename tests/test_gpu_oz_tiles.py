"""The untuned int8 tile is chosen by size (128 x 128 where the 256 x 256 grid
is short or mostly padding); every choice gives the bits of the set variant 15.
Sizes at the edges of the 128 and 256 paddings and of the rule."""
import numpy as np
import pytest

import vcp_amd

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (127, 129, 64), (128, 128, 128), (129, 256, 130), (257, 120, 65), (300, 511, 1000),
         (100, 2500, 33), (1000, 1000, 96), (1025, 1040, 70), (1300, 1280, 40), (1281, 2000, 40)]


@pytest.fixture(scope="module")
def ctx():
    return vcp_amd.Context()


def _operand(rng, m, n, width):
    a = vcp_amd.pairs(m, n)
    x = rng.standard_normal((m, n)) * np.exp2(rng.integers(-8, 9, (m, n)))
    a[..., 0] = x - np.abs(x) * width
    a[..., 1] = x + np.abs(x) * width
    return a


@pytest.mark.parametrize("m,n,k", SIZES)
def test_interval_tile_choice_keeps_bits(ctx, m, n, k):
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    A, B = _operand(rng, m, k, 2.0 ** -30), _operand(rng, k, n, 2.0 ** -35)
    ctx.set_param(vcp_amd.PARAM_OZ_VARIANT, 15)
    try:
        want = ctx.igemm(A, B, form=vcp_amd.FORM_OZAKI)
    finally:
        ctx.set_param(vcp_amd.PARAM_OZ_VARIANT, 0)
    got = ctx.igemm(A, B, form=vcp_amd.FORM_OZAKI)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("m,n,k", SIZES)
def test_dd_tile_choice_keeps_bits(ctx, m, n, k):
    rng = np.random.default_rng(m + n * 5 + k * 11)
    def dd(r, c):
        a = vcp_amd.pairs(r, c)
        a[..., 0] = rng.standard_normal((r, c))
        a[..., 1] = a[..., 0] * 2.0 ** -54 * rng.uniform(-1, 1, (r, c))
        return a
    A, B = dd(m, k), dd(k, n)
    ctx.set_param(vcp_amd.PARAM_OZ_VARIANT, 15)
    try:
        want = ctx.ddgemm(A, B)
    finally:
        ctx.set_param(vcp_amd.PARAM_OZ_VARIANT, 0)
    assert np.array_equal(ctx.ddgemm(A, B), want)
