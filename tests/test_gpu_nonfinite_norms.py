"""||R IA - I||_inf of systems with a non-finite operand end: the maximum over
the batched residual's row sums follows mats::norminf (vcp/mats.hpp:1593-1598:
row 0's NaN stays, a later row's is passed over) like the single solve's, so
a batched solve of such a system fails its verification too."""
import numpy as np
import pytest

import oracle_ffi as O
import vcp_amd
from vcp_amd import workloads as W

pytestmark = pytest.mark.gpu

# an operand end set to a value: (matrix, row, column, end, value)
ENDS = [("IA", 3, 5, 0, np.nan), ("IA", 3, 5, 1, np.nan), ("IA", 0, 0, 1, np.inf), ("IA", 4, 1, 0, -np.inf),
        ("R", 0, 2, None, np.nan)]


def _system(rng, n, end):
    R, IA = W.residual_problem(rng, n)
    name, i, j, e, v = end
    if name == "R":
        R[i, j] = v
    else:
        IA[i, j, e] = v
    return R, IA


@pytest.mark.parametrize("end", ENDS, ids=lambda e: "%s_%d%d_%s" % (e[0], e[1], e[2], e[4]))
@pytest.mark.parametrize("n", [9, 70])
def test_norm_of_non_finite_system(ctx, n, end):
    print("n", n, end, flush=True)
    rng = np.random.default_rng(n)
    R, IA = _system(rng, n, end)
    good = W.residual_problem(rng, 20)
    Ib = W.uniform_intervals(rng, n, 2, -45)
    Co, want = O.residual(R, IA)
    Cs, nub = ctx.residual_batched([good[0], R], [good[1], IA])
    assert np.array_equal(Cs[1], Co, equal_nan=True)
    # an element with one end NaN and one infinite counts as infinite here, which fails as well
    assert np.array_equal(nub[1], want, equal_nan=True) or (np.isinf(end[4]) and nub[1] == np.inf)
    assert nub[0] == O.residual(*good)[1]
    assert not want < 1.0   # every such system is one that cannot be verified
    with pytest.raises(vcp_amd.VcphipError) as single:
        ctx.lss(IA, Ib, R)
    with pytest.raises(vcp_amd.VcphipError) as batched:
        ctx.lss_batched([good[1], IA], [W.uniform_intervals(rng, 20, 1, -45), Ib], [good[0], R])
    assert single.value.code == batched.value.code == -6


def test_later_row_nan_is_passed_over(ctx):
    rng = np.random.default_rng(1)
    R, IA = W.residual_problem(rng, 40)
    R[7, 3] = np.nan   # NaN in row 7 of R IA only
    nub = ctx.residual_batched([R], [IA])[1][0]
    assert nub == O.residual(R, IA)[1] and nub < 1.0
