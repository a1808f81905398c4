"""Galerkin matrix with points where an end is infinite: operands are stored by
magnitude, and a semi-infinite negative interval of a marked point goes through
that order and its inverse in the general form.  Bit for bit the oracle."""
import numpy as np
import pytest

import oracle_ffi as O
from test_gpu_galerkin_points import _case

pytestmark = pytest.mark.gpu

KINDS = {"up": (1.0, np.inf), "down": (-np.inf, -1.0), "both": (-np.inf, np.inf), "neg0": (-np.inf, -0.5)}


@pytest.mark.parametrize("where", ["phi", "w", "u"])
@pytest.mark.parametrize("kind", sorted(KINDS))
def test_infinite_ends(ctx, where, kind):
    rng = np.random.default_rng(len(where) * 10 + len(kind))
    m, npts = 70, 83
    phi, w, u = _case(rng, m, npts)
    for k in (0, 15, 16, 47, 82):    # first and last points of stages, the last one
        if where == "phi":
            phi[rng.integers(m), k] = KINDS[kind]
        else:
            (w if where == "w" else u)[k] = KINDS[kind]
    want = O.uhphiphi(phi, w, u)
    assert np.isinf(want).any()
    assert np.array_equal(ctx.uhphiphi(phi, w, u), want, equal_nan=True)
