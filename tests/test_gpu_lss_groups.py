"""Verified solves of many right-hand sides: the enclosure is written in groups
of 64 (n / 4 from n = 257 on), a workgroup per row block and group, and the row
sums of |y| are row blocks of their own.  Bit for bit the oracle at the edges of
the groups, single and batched, and with a NaN right-hand side."""
import numpy as np
import pytest

import oracle_ffi as O
import vcp_amd
from vcp_amd import workloads as W

pytestmark = pytest.mark.gpu


def _system(n, nrhs):
    rng = np.random.default_rng(n * 1000 + nrhs)
    A = rng.uniform(-1, 1, (n, n)) + 0.5 * n * np.eye(n)
    b = rng.uniform(-1, 1, (n, nrhs))
    return (W.interval_from_midrad(A, np.ldexp(np.abs(A), -30)), W.interval_from_midrad(b, np.ldexp(np.abs(b), -30)),
            np.asfortranarray(np.linalg.inv(A)))


@pytest.mark.parametrize("n,nrhs", [(2, 200), (9, 63), (9, 64), (8, 65), (17, 129), (40, 1000), (256, 65), (257, 65),
                                    (300, 72), (300, 73), (297, 150)])
def test_groups_bitexact(ctx, n, nrhs):
    print("lss groups n=%d nrhs=%d" % (n, nrhs), flush=True)
    IA, Ib, R = _system(n, nrhs)
    Xo, go, ok = O.lss(IA, Ib, R)
    assert ok
    X, g = ctx.lss(IA, Ib, R)
    assert g == go and np.array_equal(X, Xo)
    small = _system(10, 3)
    Xb, gb = ctx.lss_batched([small[0], IA], [small[1], Ib], [small[2], R])
    assert gb[1] == go and np.array_equal(Xb[1], Xo)
    assert np.array_equal(Xb[0], O.lss(*small)[0])


def test_nan_right_hand_side(ctx):
    IA, Ib, R = _system(30, 70)
    Ib[4, 69, 1] = np.nan   # its column of y is NaN, so the norm is and every enclosure
    Xo, go, ok = O.lss(IA, Ib, R)
    assert ok and np.isnan(Xo).all()
    X, g = ctx.lss(IA, Ib, R)
    assert g == go and np.isnan(X).all()
    Xb, gb = ctx.lss_batched([IA], [Ib], [R])
    assert gb[0] == go and np.isnan(Xb[0]).all()
