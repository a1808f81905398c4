"""The tile that a plan query reports is the one the products run, whether the
size, the tuner, a saved table or a parameter chose it, and the tuner times the
128 x 128 tile (variant 7) with the padding that the products give it."""
import numpy as np
import pytest

import oracle_ffi as O
import vcp_amd
from vcp_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture
def ctx():
    c = vcp_amd.Context(0)
    yield c
    c.close()


# short grids and padded ones take variant 7, filled ones and long k 15
@pytest.mark.parametrize("m,n,k,variant", [(1, 1, 1, 7), (500, 500, 500, 7), (300, 280, 520, 7), (2048, 2048, 2048, 15),
                                           (1300, 1300, 1000, 7), (1300, 1300, 8192, 15), (100, 4000, 30000, 7),
                                           (1000, 1000, 8192, 15)])
def test_plan_reports_the_rule(ctx, m, n, k, variant):
    assert ctx.ozaki_plan(m, n, k)["variant"] == variant
    ctx.set_param(vcp_amd.PARAM_OZ_VARIANT, 9)
    assert ctx.ozaki_plan(m, n, k)["variant"] == 9
    ctx.set_param(vcp_amd.PARAM_OZ_VARIANT, 7)
    assert ctx.ozaki_plan(m, n, k)["variant"] == 7


def test_tuner_finds_the_small_tile(ctx, tmp_path):
    # 100 x 4000: half of the 256 x 256 tiles' area is padding
    m, n, k = 100, 4000, 1000
    v, ms = ctx.tune_igemm_tile(m, n, k)
    print("tuned", v, ms, flush=True)
    assert v == 7 and ms > 0.0
    assert ctx.ozaki_plan(m, n, k)["variant"] == v
    vd, _ = ctx.tune_ddgemm_tile(m, n, k)
    assert vd == 7
    path = str(tmp_path / "tune.txt")
    ctx.tune_save(path)
    with vcp_amd.Context(0) as c2:
        c2.tune_load(path)
        assert c2.ozaki_plan(m, n, k)["variant"] == v


@pytest.mark.parametrize("line,variant", [("igemm 11 11 11 7 16 1", 10), ("igemm 11 11 11 7 16 1 128", 7),
                                          ("igemm 11 11 11 7 16 1 256", 10), ("igemm 11 11 11 9 16 1", 9),
                                          ("igemm 11 11 11 7 16", 10)])
def test_tables_of_the_older_seven(ctx, tmp_path, line, variant):
    # 7 stood for 128 x 256 tiles, which are variant 10's, before it was the 128 x 128 tile
    path = tmp_path / "tune.txt"
    path.write_text("vcphip-tune %d\n%s\n" % (1 if len(line.split()) == 6 else 2, line))
    ctx.tune_load(str(path))
    assert ctx.ozaki_plan(2000, 2000, 2000)["variant"] == variant
    again = tmp_path / "again.txt"
    ctx.tune_save(str(again))
    with vcp_amd.Context(0) as c2:
        c2.tune_load(str(again))
        assert c2.ozaki_plan(2000, 2000, 2000)["variant"] == variant


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (130, 257, 65), (300, 511, 200)])
def test_set_small_tile_bits(ctx, m, n, k):
    rng = np.random.default_rng(m + n + k)
    A, B = W.wide_exponent_intervals(rng, m, k), W.wide_exponent_intervals(rng, k, n)
    ctx.set_param(vcp_amd.PARAM_OZ_VARIANT, 7)
    assert np.array_equal(ctx.igemm(A, B, vcp_amd.FORM_OZAKI), O.ozaki_igemm(A, B, 16))
