"""The plain product of one column at more rows than a launch of the row-serial
form holds (fewer than 2^32 threads): exact products of small whole numbers."""
import pytest
import torch

import vcp_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [(1 << 26) - 1, 1 << 26, (1 << 27) + 9])
def test_tall_product(ctx, m):
    print("tall m", m, flush=True)
    A = torch.arange(m, device="cuda", dtype=torch.float64) % 1021 - 500
    B = torch.full((1,), 3.0, dtype=torch.float64, device="cuda")
    U, D = torch.zeros_like(A), torch.zeros_like(A)
    torch.cuda.synchronize()
    own = vcp_amd.Context()   # its workspace (17 GB of planes) goes with it
    try:
        own.gemm_rurd_dev(m, 1, 1, A.data_ptr(), m, B.data_ptr(), 1, U.data_ptr(), D.data_ptr(), m)
        own.synchronize()
    finally:
        own.close()
    assert torch.equal(U, A * 3.0) and torch.equal(D, A * 3.0)
