"""A factorisation that fails leaves the rows below its last diagonal block as
they were: the wavefront that factors a block writes no rows but its own."""
import numpy as np
import pytest
import torch

from gputils_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [40, 64, 100, 128])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_rows_below_the_diagonal_block(n, dtype):
    M = np.random.default_rng(n).standard_normal((n, n))
    A = M @ M.T + n * np.eye(n)
    A[20, 20] = -1e6  # the second block of 16 fails
    t = torch.from_numpy(A[None]).to(dtype).cuda()
    was = t.clone()
    assert api.potrf_batched(t).item() == 21
    L = np.linalg.cholesky(A[:16, :16])
    got = t[0].double().cpu().numpy().T
    assert np.abs(np.tril(got[:16, :16]) - L).max() <= 1e-5 * np.abs(L).max()
    assert torch.equal(t[0, :16, 16:], was[0, :16, 16:])
