"""Cholesky of n > 128 outside the normal range: subnormal pivots in FP32,
infinite diagonal entries (a variable held at zero by a penalty), a factor
whose diagonal has no normal reciprocal."""
import numpy as np
import pytest
import torch

from gputils_amd import api

pytestmark = pytest.mark.gpu

SIZES = [129, 225, 513]  # two, four and six strips a wavefront; a last block of one row


def spd(n):
    M = np.random.default_rng(n).standard_normal((n, n))
    return M @ M.T / n + np.eye(n)


def put(M, dtype):
    return torch.from_numpy(np.ascontiguousarray(M.T)[None]).to(dtype).cuda()


@pytest.mark.parametrize("n", SIZES)
def test_subnormal_pivots(n):
    """L L^T = A: every step rounds at the size of A in FP32, or at the smallest subnormal."""
    t = put(spd(n) * 1e-39, torch.float32)
    A = t[0].double().cpu().numpy()
    assert api.potrf_batched(t).item() == 0
    L = np.tril(t[0].double().cpu().numpy().T)
    assert np.isfinite(L).all()
    assert np.abs(L @ L.T - A).max() <= 2 * n * (2.0 ** -149 + 2.0 ** -23 * np.abs(A).max())


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_infinite_diagonal(n, dtype):
    """The factor and solution are those without these rows and columns
    (condition number near 5: n eps kappa, as for the other factor tests)."""
    tol = 2e-4 if dtype == torch.float32 else 1e-12
    out = [0, 50, n - 1]
    keep = np.setdiff1d(np.arange(n), out)
    A = spd(n)
    for k in out:
        A[k, k] = np.inf
    B = np.random.default_rng(1).standard_normal((n, 5))
    t, b = put(A, dtype), put(B, dtype)
    assert api.potrf_batched(t).item() == 0
    api.potrs_batched(t, b)
    L, X = np.tril(t[0].double().cpu().numpy().T), b[0].double().cpu().numpy().T
    assert np.isinf(L[out, out]).all()
    for k in out:
        assert (L[k + 1:, k] == 0).all()
    ref = np.linalg.cholesky(A[np.ix_(keep, keep)])
    assert np.abs(L[np.ix_(keep, keep)] - ref).max() <= tol * np.abs(ref).max()
    x = np.linalg.solve(A[np.ix_(keep, keep)], B[keep])
    assert np.abs(X[keep] - x).max() <= tol * np.abs(x).max() and (X[out] == 0).all()


@pytest.mark.parametrize("n", SIZES + [672])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_factor_without_normal_reciprocals(n, dtype):
    """Two rows of their own with a subnormal diagonal entry d: x is b / d / d
    there (0, or a finite quotient), and b / 4 elsewhere; three roundings."""
    eps = torch.finfo(dtype).eps
    d = float(torch.tensor(1e-39 if dtype == torch.float32 else 1e-309, dtype=dtype))
    least = 2.0 ** -149 if dtype == torch.float32 else 2.0 ** -1074
    L = np.eye(n) * 2
    L[7, 7] = L[n - 1, n - 1] = d
    B = np.random.default_rng(n).uniform(1, 2, (n, 5))
    B[7] = [0.0, least, -least, 0.0, 3 * least]
    B[n - 1] = [least, 0.0, 0.0, 2 * least, 0.0]
    t, b = put(L, dtype), put(B, dtype)
    B = b[0].double().cpu().numpy().T
    api.potrs_batched(t, b)
    X = b[0].double().cpu().numpy().T
    want = B / np.diag(L)[:, None] / np.diag(L)[:, None]
    assert np.isfinite(X).all()
    assert (np.abs(X - want) <= 3 * eps * np.abs(want)).all()
