"""dd products of k = 0 on device pointers, where an operand without elements
may have no memory: zeros, whatever earlier products left in the workspace."""
import pytest
import torch

import vcp_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["vcphip_ddgemm_dev", "vcphip_ddgemm_ta_dev"])
@pytest.mark.parametrize("null", ["A", "B", "both", "none"])
@pytest.mark.parametrize("m,n", [(1, 1), (10, 23), (300, 17)])
def test_dd_product_of_nothing(ctx, m, n, null, name):
    call = getattr(vcp_amd.lib(), name)
    # an earlier product leaves exponents 2 and 3 where the flags of this one go (2: a non-finite row)
    X = torch.rand((300, 300, 2), dtype=torch.float64, device="cuda") * 2.0 + 1.0
    Y = torch.zeros_like(X)
    C = torch.full((n, m, 2), 7.0, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    assert call(ctx._h, 300, 300, 300, X.data_ptr(), 300, X.data_ptr(), 300, Y.data_ptr(), 300) == 0
    a = None if null in ("A", "both") else X.data_ptr()
    b = None if null in ("B", "both") else X.data_ptr()
    assert call(ctx._h, m, n, 0, a, m if name == "vcphip_ddgemm_dev" else 1, b, 1, C.data_ptr(), m) == 0
    ctx.synchronize()
    assert (C == 0.0).all()
