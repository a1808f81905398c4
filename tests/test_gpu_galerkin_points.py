"""Galerkin matrix at the edges of its 32-row tiles and 16-point stages, with
points where single elements hold zero, an end is infinite or an end is zero
next to points in the two-product form: bit-identical to the oracle."""
import numpy as np
import pytest

import oracle_ffi as O
from vcp_amd import workloads as W

pytestmark = pytest.mark.gpu


def _case(rng, m, npts):
    phi = W.uniform_intervals(rng, m, npts, -30)
    w = W.uniform_intervals(rng, 1, npts, -40)[0]
    u = W.uniform_intervals(rng, 1, npts, -35)[0]
    return phi, np.ascontiguousarray(w), np.ascontiguousarray(u)


@pytest.mark.parametrize("m", [1, 31, 32, 33, 64, 97])
@pytest.mark.parametrize("npts", [1, 15, 16, 17, 32, 33, 49])
def test_tile_and_stage_edges(ctx, m, npts):
    phi, w, u = _case(np.random.default_rng(100 * m + npts), m, npts)
    assert np.array_equal(ctx.uhphiphi(phi, w, u), O.uhphiphi(phi, w, u))


@pytest.mark.parametrize("where", ["phi", "w", "u"])
@pytest.mark.parametrize("kind", ["straddle", "zero", "lo0", "hi0"])
def test_single_points_outside_the_two_product_form(ctx, where, kind):
    rng = np.random.default_rng(len(where) * 10 + len(kind))
    m, npts = 70, 83
    phi, w, u = _case(rng, m, npts)
    value = {"straddle": (-0.25, 0.5), "zero": (0.0, 0.0), "lo0": (0.0, 0.5), "hi0": (-0.5, 0.0)}[kind]
    for k in (0, 15, 16, 40, 47, 79, 82):    # first and last points of stages, the last one
        if where == "phi":
            phi[rng.integers(m), k] = value
        else:
            (w if where == "w" else u)[k] = value
    assert np.array_equal(ctx.uhphiphi(phi, w, u), O.uhphiphi(phi, w, u))
