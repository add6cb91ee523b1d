"""Least squares over several launches, whose reflector scalars are formed
again from the reflectors: columns whose tail is nonzero while the square of
the scaled tail underflows.  Such a reflector still turns the sign of its row
(tau = 2), for the columns right of its panel and for the right-hand sides too.

The systems are Gaussian but for that one column, so the factorisation, which
does not see the columns' scales, solves to 20 n eps (n <= 65): 2e-4 in FP32
and 1e-11 in FP64, of the largest component."""
import numpy as np
import pytest
import torch

from gputils_amd import api

pytestmark = pytest.mark.gpu

# down to tails whose own square underflows (H = I) and to zero
TAILS = {torch.float32: [1e-15, 1e-18, 1e-21, 3e-23, 1e-26, 0.0],
         torch.float64: [1e-130, 1e-150, 1e-160, 1e-164, 0.0]}


def _solve(A, B, dtype):
    """A (m, n), B (m, nrhs) -> the solution and R, with the inputs as the type holds them."""
    ta = torch.from_numpy(np.ascontiguousarray(A.T)[None]).to(dtype).cuda()
    tb = torch.from_numpy(np.ascontiguousarray(B.T)[None]).to(dtype).cuda()
    A, B = ta[0].double().cpu().numpy().T, tb[0].double().cpu().numpy().T
    api.gels_batched(ta, tb)
    n = A.shape[1]
    return A, B, tb[0].double().cpu().numpy().T[:n], np.triu(ta[0].double().cpu().numpy().T[:n])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("m,n,nrhs", [(300, 40, 2), (40, 24, 300), (1024, 65, 1)])
@pytest.mark.parametrize("col,alpha", [(0, 1e3), (0, -1.0), (17, 1e3)])
def test_vanishing_tail(m, n, nrhs, col, alpha, dtype):
    """Column `col` starts at row `col` with alpha, the columns before it are
    triangular (their reflectors are the identity); in the first panel and the second."""
    r = np.random.default_rng(m + col)
    tol = 2e-4 if dtype == torch.float32 else 1e-11
    for tail in TAILS[dtype]:
        A, B = r.standard_normal((m, n)), r.standard_normal((m, nrhs))
        A[:, :col] = 0
        A[:col, :col] = np.triu(r.standard_normal((col, col)), 1) * 0.1 + 2 * np.eye(col)
        A[col, col], A[col + 1:, col] = alpha, tail
        A, B, X, R = _solve(A, B, dtype)
        ref = np.linalg.lstsq(A, B, rcond=None)[0]
        assert np.max(np.abs(X - ref)) <= tol * np.abs(ref).max(), tail
        # R as the one-launch form has it, signs included
        one = torch.from_numpy(np.ascontiguousarray(A.T)[None]).to(dtype).cuda()
        api.geqrf_batched(one)
        one = np.triu(one[0].double().cpu().numpy().T[:n])
        assert np.max(np.abs(R - one)) <= tol * np.abs(one).max(), tail
