"""Infinities and NaNs in QR, least squares and Q application: a reflector
reads and changes the rows from its own on, H = I (tau = 0) none, as in
LAPACK's unblocked algorithm, which the model below follows.  Entries that the
model leaves finite are finite, with its value (n eps times a condition number
near 20, as in the other QR tests: 2e-4 in FP32, 1e-11 in FP64)."""
import numpy as np
import pytest
import torch

from gputils_amd import api

pytestmark = pytest.mark.gpu

# one launch with 16 lanes a column, panels, whole wavefronts, one slot more than a panel
SHAPES = [(20, 8), (40, 40), (100, 30), (256, 129), (300, 40), (700, 20)]


def qr_model(A):
    A = A.copy()
    m, n = A.shape
    tau = np.zeros(n)
    for j in range(n):
        sq = float((A[j + 1:, j] ** 2).sum())
        if sq != 0.0:
            norm = np.sqrt(A[j, j] ** 2 + sq)
            beta = -norm if A[j, j] >= 0 else norm
            tau[j] = (beta - A[j, j]) / beta
            A[j + 1:, j] *= 1.0 / (A[j, j] - beta)
            A[j, j] = beta
            if tau[j] != 0.0:
                v = np.concatenate([[1.0], A[j + 1:, j]])
                for c in range(j + 1, n):
                    A[j:, c] -= tau[j] * (v @ A[j:, c]) * v
    return A, tau


def apply_model(A, tau, x, trans):
    x = x.copy()
    n = A.shape[1]
    for j in (range(n) if trans else range(n - 1, -1, -1)):
        if tau[j] != 0.0:
            v = np.concatenate([[1.0], A[j + 1:, j]])
            x[j:] -= tau[j] * (v @ x[j:]) * v
    return x


def close(got, want, tol):
    ok = np.isfinite(want)
    assert np.isfinite(got[ok]).all()
    assert not np.isfinite(got[~ok]).any()
    assert np.max(np.abs(got[ok] - want[ok]), initial=0) <= tol * np.max(np.abs(want[ok]), initial=1)


def put(M, dtype):
    return torch.from_numpy(np.ascontiguousarray(np.swapaxes(M, -1, -2))[None]).to(dtype).cuda()


def matrices(m, n, dtype):
    r = np.random.default_rng(m + n)
    full = r.standard_normal((m, n))
    tri = np.zeros((m, n))
    tri[:n] = np.triu(r.standard_normal((n, n))) + 4 * np.eye(n)
    mixed = tri.copy()
    mixed[n // 2:, n // 2:] = r.standard_normal((m - n // 2, n - n // 2))  # H = I for the first half
    f = lambda M: torch.from_numpy(M).to(dtype).double().numpy()  # noqa: E731
    for name, M, at in (("full", full, (3, n // 2)), ("triangular", tri, (1, n - 1)), ("mixed", mixed, (1, n - 1))):
        for bad in (np.inf, np.nan):
            B = f(M)
            B[at] = bad
            yield f"{name} {bad}", B


@pytest.mark.filterwarnings("ignore::RuntimeWarning")
@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_factors(m, n, dtype):
    tol = 2e-4 if dtype == torch.float32 else 1e-11
    for name, A in matrices(m, n, dtype):
        want, tau0 = qr_model(A)
        t = put(A, dtype)
        tau = api.geqrf_batched(t)[0].double().cpu().numpy()
        print(name, flush=True)
        got = t[0].double().cpu().numpy().T
        # R row by row and the finite reflectors; a NaN column's own entries are NaN in both
        close(np.triu(got[:n]), np.triu(want[:n]), tol)
        fin = np.isfinite(tau0)
        close(got[:, fin], want[:, fin], tol)
        close(tau, tau0, tol)


@pytest.mark.filterwarnings("ignore::RuntimeWarning")
@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_q_application_and_least_squares(m, n, dtype):
    """An infinity in one column of C, or of the right-hand sides: the others
    come out as without it; rows that no reflector joins to it stay finite."""
    tol = 2e-4 if dtype == torch.float32 else 1e-11
    r = np.random.default_rng(m * n)
    A = np.zeros((m, n))
    A[:n] = np.triu(r.standard_normal((n, n)), 1) / n + 4 * np.eye(n)
    A[n // 2:, n // 2:] = r.standard_normal((m - n // 2, n - n // 2))
    A = torch.from_numpy(A).to(dtype).double().numpy()
    h, tau0 = qr_model(A)
    C = torch.from_numpy(r.standard_normal((m, 3))).to(dtype).double().numpy()
    C[1, 1] = np.inf
    t, c = put(A, dtype), put(C, dtype)
    tau = api.geqrf_batched(t)
    for trans in (True, False):
        got = api.ormqr_batched(t, tau, c.clone(), trans=trans)[0].double().cpu().numpy().T
        for q in range(3):
            close(got[:, q], apply_model(h, tau0, C[:, q], trans), tol)
    a, b = put(A, dtype), put(C, dtype)
    api.gels_batched(a, b)
    got = b[0].double().cpu().numpy().T
    for q in range(3):
        y = apply_model(h, tau0, C[:, q], True)[:n]
        for k in range(n - 1, -1, -1):
            y[k] /= h[k, k]
            y[:k] -= h[:k, k] * y[k]
        close(got[:n, q], y, tol)
    assert np.array_equal(got[n:], C[n:])
