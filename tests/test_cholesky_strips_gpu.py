"""Cholesky of n > 128: the strip kernels against the FP64 oracle at the edges
of their ranges (a last block of one row, full blocks, the slot counts 2 | 4 |
6, one | two rows per thread of the solve, the first n of the global path).

A = M M^T + n I has a condition number near 5, so the factor and the
solution agree with the oracle to n eps kappa: 672 * 1.1e-16 * 5 < 1e-12 in
FP64 and 672 * 6e-8 * 5 = 2e-4 in FP32."""
import ctypes

import numpy as np
import pytest
import torch

from gputils_amd import api
from gputils_amd._lib import lib

pytestmark = pytest.mark.gpu

EDGES = [129, 144, 207, 224, 225, 448, 449, 512, 513, 657, 672, 673]


def spd(k, n, seed):
    M = np.random.default_rng(seed).standard_normal((k, n, n))
    return M @ np.swapaxes(M, 1, 2) + n * np.eye(n)


@pytest.mark.parametrize("n", EDGES)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_factor_and_solve_with_padding(oracle, n, dtype):
    """lda = n + 3, ldb = n + 1; the strictly upper part and the padding
    hold NaN: never used, left as they are."""
    k, nrhs, lda, ldb = 2, 5, n + 3, n + 1
    A = spd(k, n, n)
    B = np.random.default_rng(n + 1).standard_normal((k, nrhs, n))
    a = np.full((k, n, lda), np.nan)
    b = np.full((k, nrhs, ldb), np.nan)
    low = np.tril(np.ones((n, n), bool))
    for i in range(k):
        a[i, :, :n] = np.where(low, A[i], np.nan).T
    b[:, :, :n] = B
    ta, tb = torch.from_numpy(a).to(dtype).cuda(), torch.from_numpy(b).to(dtype).cuda()
    info = torch.full((k,), -7, dtype=torch.int32, device="cuda")
    p = "d" if dtype == torch.float64 else "s"
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    st = api.stream_handle()
    assert getattr(lib(), f"gputils_{p}potrf_batched")(n, P(ta), lda, n * lda, P(info), k, st) == 0
    assert info.cpu().tolist() == [0] * k
    assert getattr(lib(), f"gputils_{p}potrs_batched")(n, nrhs, P(ta), lda, n * lda, P(tb), ldb, nrhs * ldb,
                                                       P(info), k, st) == 0
    La, X = ta.cpu().double().numpy(), tb.cpu().double().numpy()
    tol = 1e-12 if dtype == torch.float64 else 2e-4
    for i in range(k):
        L, oinfo = oracle.potrf(A[i])
        assert oinfo == 0
        got = La[i, :, :n].T
        assert np.max(np.abs(got[low] - np.tril(L)[low])) <= tol * np.abs(L).max()
        assert np.isnan(got[~low]).all() and np.isnan(La[i, :, n:]).all()
        ref = np.linalg.solve(A[i], B[i].T).T
        assert np.max(np.abs(X[i, :, :n] - ref)) <= tol * np.abs(ref).max()
        assert np.isnan(X[i, :, n:]).all()


@pytest.mark.parametrize("n", [129, 225, 672])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_failing_minor(oracle, n, dtype):
    """Indefinite, zero and NaN pivots in the first, a middle and the last
    block: the oracle's info, and the neighbours factorise."""
    k = 5
    A = spd(k, n, 3 * n)
    A[0][0, 0] = 0.0
    A[1][n // 2, n // 2] = -1e6
    A[3][n - 1, n - 1] = -1e6
    A[4][70, 70] = np.nan
    t = torch.from_numpy(np.ascontiguousarray(np.swapaxes(A, 1, 2))).to(dtype).cuda()
    info = api.potrf_batched(t).cpu().tolist()
    assert info == [1, n // 2 + 1, 0, n, 71]
    L, _ = oracle.potrf(A[2])
    got = api.to_matrices(t).cpu().double().numpy()[2]
    assert np.max(np.abs(np.tril(got) - np.tril(L))) <= (1e-12 if dtype == torch.float64 else 2e-4) * np.abs(L).max()
