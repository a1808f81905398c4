"""Few columns of many rows: the row-serial form is taken up to a number of row
blocks that depends on the columns, the form and k, the planes beyond it.  The
route as the stage times name it (a product from planes times them), and the
bits of both forms, which a forced tile height makes equal."""
import pytest
import torch

import vcp_amd

pytestmark = pytest.mark.gpu

# form, n, k, row blocks of 8 per CU at which the row-serial form ends (None: it never does)
RULES = [("ii", 8, 16, 16), ("pp", 8, 63, 16), ("pi", 8, 64, None), ("ip", 9, 32, 8), ("pi", 16, 63, 8),
         ("ii", 16, 64, None), ("ii", 17, 200, 3), ("pi", 32, 16, 3), ("ip", 17, 127, 16), ("pp", 32, 16, 16),
         ("ip", 32, 128, None)]


def _call(c, form, m, n, k, A, B, C, C2):
    L, P = vcp_amd.lib(), lambda t: t.data_ptr()
    if form == "ii":
        rc = L.vcphip_igemm_dev(c.handle, vcp_amd.FORM_PLAIN, m, n, k, P(A), m, P(B), k, P(C), m)
    elif form == "ip":
        rc = L.vcphip_igemm_ip_dev(c.handle, m, n, k, P(A), m, P(B), k, P(C), m)
    elif form == "pi":
        rc = L.vcphip_igemm_pi_dev(c.handle, m, n, k, P(A), m, P(B), k, P(C), m)
    else:
        rc = L.vcphip_gemm_rurd_dev(c.handle, m, n, k, P(A), m, P(B), k, P(C), P(C2), m, 0)
    assert rc == 0
    c.synchronize()


@pytest.mark.parametrize("over", [0, 1])
@pytest.mark.parametrize("form,n,k,limit", RULES)
def test_route_and_bits(form, n, k, limit, over):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    m = 8 * cus * (limit or 17) + (1 if over else 0)
    print("rows %s m=%d n=%d k=%d" % (form, m, n, k), flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = lambda r, c, iv: (torch.rand((c, r, 2) if iv else (c, r), dtype=torch.float64, device="cuda",  # noqa: E731
                                     generator=g) - 0.5)
    A, B = x(m, k, form[0] == "i"), x(k, n, form[1] == "i")
    for t in (A, B):
        if t.dim() == 3:
            t.copy_(t.sort(dim=-1)[0])
    outs = []
    with vcp_amd.Context(0) as c:
        for rows in (0, 64):
            c.set_param(vcp_amd.PARAM_PLANE_ROWS, rows)
            c.set_param(vcp_amd.PARAM_STAGE_TIMING, 1)
            C = torch.full((n, m, 1 if form == "pp" else 2), 7.0, dtype=torch.float64, device="cuda")
            C2 = torch.full((n, m), 7.0, dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            _call(c, form, m, n, k, A, B, C, C2)
            assert ("planes" in c.stage_times()) == bool(rows or (limit and over))
            outs.append((C, C2))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
