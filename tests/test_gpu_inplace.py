"""Plain single products whose result lies over an operand, on device pointers:
A <- A B and B <- A B (whole, or shifted so that the ranges only overlap), at
sizes on both sides of the rule between the row-serial form, which reads its
operands while it stores, and the planes, which copy them first.  Bit for bit
the oracle's product of the original operands."""
import numpy as np
import pytest
import torch

import oracle_ffi as O
import vcp_amd
from vcp_amd import workloads as W
from test_gpu_planes import _dev_iv, _dev_pt, _ok, _read_iv, _wide

pytestmark = pytest.mark.gpu

# (rows of C, columns of C, which operand C replaces): few columns, small
# squares of one and of several column groups, and sizes that take tiles anyway
CASES = [(200, 5, "B"), (1000, 24, "A"), (1000, 24, "B"), (96, 96, "A"), (256, 256, "A"), (256, 256, "B"),
         (400, 400, "A"), (400, 400, "B")]


# (an interval result does not fit over a point operand)
@pytest.mark.parametrize("form,m,n,over", [(f, *c) for f in ("ii", "ip", "pi", "pp") for c in CASES
                                           if (f, c[2]) not in (("ip", "B"), ("pi", "A"))])
def test_result_over_operand(ctx, form, m, n, over):
    print("inplace %s m=%d n=%d over %s" % (form, m, n, over), flush=True)
    k = n if over == "A" else m
    rng = np.random.default_rng(m * 31 + n)
    wide = {"i": lambda r, c: W.wide_exponent_intervals(rng, r, c, rad_exp=-20), "p": lambda r, c: _wide(rng, r, c)}
    dev = {"i": _dev_iv, "p": _dev_pt}
    A, B = wide[form[0]](m, k), wide[form[1]](k, n)
    dA, dB = dev[form[0]](A, m), dev[form[1]](B, k)
    C = (dA if over == "A" else dB).data_ptr()
    L = vcp_amd.lib()
    torch.cuda.synchronize()
    if form == "pp":
        other = torch.zeros((n, m), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        _ok(L.vcphip_gemm_rurd_dev(ctx._h, m, n, k, dA.data_ptr(), m, dB.data_ptr(), k, other.data_ptr(), C, m, 0),
            "gemm_rurd_dev")   # the round-down result over the operand
        ctx.synchronize()
        up, dn = O.rgemm(A, B, 1), O.rgemm(A, B, -1)
        assert np.array_equal(other.cpu().numpy().T, up)
        assert np.array_equal((dA if over == "A" else dB).cpu().numpy().T, dn)
        return
    want = {"ii": O.pidblas_mulmm, "ip": O.pidblas_mul_im_m, "pi": O.pidblas_mul_m_im}[form](A, B)
    if form == "ii":
        rc = L.vcphip_igemm_dev(ctx._h, vcp_amd.FORM_PLAIN, m, n, k, dA.data_ptr(), m, dB.data_ptr(), k, C, m)
    elif form == "ip":
        rc = L.vcphip_igemm_ip_dev(ctx._h, m, n, k, dA.data_ptr(), m, dB.data_ptr(), k, C, m)
    else:
        rc = L.vcphip_igemm_pi_dev(ctx._h, m, n, k, dA.data_ptr(), m, dB.data_ptr(), k, C, m)
    _ok(rc, form)
    ctx.synchronize()
    assert np.array_equal(_read_iv(dA if over == "A" else dB, m), want)


@pytest.mark.parametrize("shift", [-1, 1])
def test_result_one_element_into_operand(ctx, shift):
    # C begins one column before or after B in one allocation: the ranges overlap, the starts differ
    m = k = 120
    n = 6
    rng = np.random.default_rng(5)
    A, B = _wide(rng, m, k), W.wide_exponent_intervals(rng, k, n, rad_exp=-20)
    buf = torch.zeros((n + 2, k, 2), dtype=torch.float64, device="cuda")
    buf[1:n + 1] = _dev_iv(B, k)
    dA = _dev_pt(A, m)
    torch.cuda.synchronize()
    C = buf[1 + shift:]
    _ok(vcp_amd.lib().vcphip_igemm_pi_dev(ctx._h, m, n, k, dA.data_ptr(), m, buf[1:].data_ptr(), k, C.data_ptr(), m),
        "igemm_pi_dev")
    ctx.synchronize()
    assert np.array_equal(_read_iv(C[:n], m), O.pidblas_mul_m_im(A, B))


@pytest.mark.parametrize("ka", [40, 39])
def test_row_blocks_of_one_matrix(ka):
    # B (rows 0 .. k) and C (the rows after them, or from B's last row on) in one matrix's columns
    m, n, k = 50, 6, 40
    rng = np.random.default_rng(6)
    A, B = _wide(rng, m, k), W.wide_exponent_intervals(rng, k, n, rad_exp=-20)
    ld = 100
    buf = torch.zeros((n, ld, 2), dtype=torch.float64, device="cuda")
    buf[:, :k] = _dev_iv(B, k)
    dA = _dev_pt(A, m)
    with vcp_amd.Context(0) as c:
        c.set_param(vcp_amd.PARAM_STAGE_TIMING, 1)
        torch.cuda.synchronize()
        C = buf.data_ptr() + 16 * ka
        _ok(vcp_amd.lib().vcphip_igemm_pi_dev(c.handle, m, n, k, dA.data_ptr(), m, buf.data_ptr(), ld, C, ld), "pi")
        c.synchronize()
        assert ("planes" in c.stage_times()) == (ka < k)   # apart: the row-serial form; overlapping: the planes
    assert np.array_equal(buf[:, ka:ka + m].cpu().numpy().transpose(1, 0, 2), O.pidblas_mul_m_im(A, B))
