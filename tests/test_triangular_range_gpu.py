"""Triangular solves whose diagonal holds numbers without a normal reciprocal
(subnormal ones, where it overflows, and the largest): quotients that are
finite come out finite, to the type's rounding."""
import numpy as np
import pytest
import torch

from gputils_amd import api

pytestmark = pytest.mark.gpu

F = {torch.float32: (1e-40, 3e-40, 1.5e38, 1e-6), torch.float64: (1e-310, 3e-310, 1.2e308, 1e-12)}


def triangle(n, at, d, upper):
    R = np.triu(np.random.default_rng(n).standard_normal((n, n)), 1) * 0.1 / n + 2 * np.eye(n)
    R[at, :] = R[:, at] = 0  # row and column `at` hold the diagonal entry alone
    R[at, at] = d
    return R if upper else R.T


def put(M, dtype):
    return torch.from_numpy(np.ascontiguousarray(np.swapaxes(M, -1, -2))[None]).to(dtype).cuda()


def check(X, R, B, tol):
    """X = R^{-1} B row by row, every row by its own size."""
    ref = np.array(B, dtype=np.longdouble)
    n = R.shape[0]
    for k in range(n - 1, -1, -1):
        ref[k] /= R[k, k]
        ref[:k] -= np.outer(R[:k, k], ref[k])
    assert np.isfinite(X).all()
    assert np.max(np.abs(X - ref) / np.abs(ref).max(axis=1, keepdims=True)) <= tol * n


@pytest.mark.parametrize("n", [5, 64, 100, 150, 400])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_upper_triangle(n, dtype):
    tiny, rhs, huge, tol = F[dtype]
    for d, b in ((tiny, rhs), (huge, 1.0)):
        R = triangle(n, 3, d, True)
        B = np.random.default_rng(7).uniform(1, 2, (n, 3))
        B[3] = b * np.array([1.0, 2.0, -1.0])
        t, x = put(R, dtype), put(B, dtype)
        R, B = (v[0].double().cpu().numpy().T for v in (t, x))
        x2 = torch.zeros(1, 3, n + 20, dtype=dtype, device="cuda")
        x2[:, :, :n] = x
        api.trsm_upper_batched(t, x)
        check(x[0].double().cpu().numpy().T, R, B, tol)
        # the same triangle as the factor of a least-squares problem (H = I)
        a = torch.zeros(1, n, n + 20, dtype=dtype, device="cuda")
        a[:, :, :n] = t
        api.gels_batched(a, x2)
        check(x2[0, :, :n].double().cpu().numpy().T, R, B, tol)
