"""QR, least squares, Q application and the triangular solve at the edges of
the register kernels' shapes: rows 16 KR and 64 KR and one more, the column
bins 16 | 32 | 48 | 64 | 96 | 128, panels of 16 with and without a remainder,
and the first sizes of the general kernels.

Against numpy in 64 bits.  The matrices are Gaussian with m >= 1.3 n, so their
condition number stays below about 20: a factorisation's backward error of
n eps gives factors and solutions to 20 n eps < 1e-11 in FP64 and, for n up
to 150, 20 * 150 * 6e-8 = 2e-4 in FP32."""
import ctypes

import numpy as np
import pytest
import torch

from gputils_amd import api
from gputils_amd._lib import lib

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (2, 1), (32, 16), (33, 17), (64, 32), (65, 33), (100, 48), (112, 49), (113, 64), (160, 65), (161, 96),
          (200, 97), (256, 128), (256, 129), (257, 16), (300, 17), (384, 80), (385, 81), (640, 48), (641, 20),
          (1024, 65), (1025, 12)]


def _tol(dtype):
    return 1e-11 if dtype == torch.float64 else 2e-4


def _P(t):
    return ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_qr_and_least_squares(m, n, dtype):
    """Padded leading dimensions (the padding holds NaN and stays)."""
    k, nrhs, lda, ldb = 3, 2, m + 2, m + 1
    r = np.random.default_rng(m * 1000 + n)
    A, B = r.standard_normal((k, m, n)), r.standard_normal((k, m, nrhs))
    a, b = np.full((k, n, lda), np.nan), np.full((k, nrhs, ldb), np.nan)
    a[:, :, :m], b[:, :, :m] = np.swapaxes(A, 1, 2), np.swapaxes(B, 1, 2)
    p = "d" if dtype == torch.float64 else "s"
    st, tol = api.stream_handle(), _tol(dtype)
    f = lambda x: torch.from_numpy(x).to(dtype).cuda()  # noqa: E731
    h, tau0 = np.linalg.qr(A, mode="raw")
    Q, R = np.linalg.qr(A, mode="complete")
    QtB = np.swapaxes(Q, 1, 2) @ B
    X0 = np.linalg.solve(R[:, :n], QtB[:, :n])

    ta, tb = f(a), f(b)
    tau, info = torch.zeros(k, n, dtype=dtype, device="cuda"), torch.full((k,), 5, dtype=torch.int32, device="cuda")
    assert getattr(lib(), f"gputils_{p}geqrf_batched")(m, n, _P(ta), lda, n * lda, _P(tau), n, _P(info), k, st) == 0
    got = ta.cpu().double().numpy()
    assert info.cpu().tolist() == [0] * k
    assert np.max(np.abs(got[:, :, :m] - h)) <= tol * np.abs(h).max() and np.isnan(got[:, :, m:]).all()
    assert np.max(np.abs(tau.cpu().double().numpy() - tau0)) <= tol * 2
    # Q^T B, then Q (Q^T B) = B
    assert getattr(lib(), f"gputils_{p}ormqr_batched")(1, m, nrhs, n, _P(ta), lda, n * lda, _P(tau), n, _P(tb), ldb,
                                                       nrhs * ldb, k, st) == 0
    c = np.swapaxes(tb.cpu().double().numpy()[:, :, :m], 1, 2)
    assert np.max(np.abs(c - QtB)) <= tol * np.abs(QtB).max()
    t2 = tb.clone()
    assert getattr(lib(), f"gputils_{p}ormqr_batched")(0, m, nrhs, n, _P(ta), lda, n * lda, _P(tau), n, _P(t2), ldb,
                                                       nrhs * ldb, k, st) == 0
    c = np.swapaxes(t2.cpu().double().numpy()[:, :, :m], 1, 2)
    assert np.max(np.abs(c - B)) <= tol * np.abs(B).max()
    # R^{-1} (Q^T B)
    assert getattr(lib(), f"gputils_{p}trsm_upper_batched")(n, nrhs, _P(ta), lda, n * lda, _P(tb), ldb, nrhs * ldb,
                                                            k, st) == 0
    c = np.swapaxes(tb.cpu().double().numpy(), 1, 2)
    assert np.max(np.abs(c[:, :n] - X0)) <= tol * np.abs(X0).max()
    assert np.max(np.abs(c[:, n:m] - QtB[:, n:]), initial=0) <= tol * np.abs(QtB).max()
    # the same in one call: factors over A, the solution over B's first rows
    ta, tb = f(a), f(b)
    assert getattr(lib(), f"gputils_{p}gels_batched")(m, n, nrhs, _P(ta), lda, n * lda, _P(tb), ldb, nrhs * ldb,
                                                      _P(info), k, st) == 0
    got, c = ta.cpu().double().numpy(), np.swapaxes(tb.cpu().double().numpy(), 1, 2)
    assert np.max(np.abs(got[:, :, :m] - h)) <= tol * np.abs(h).max() and np.isnan(got[:, :, m:]).all()
    assert np.max(np.abs(c[:, :n] - X0)) <= tol * np.abs(X0).max()
    assert np.array_equal(c[:, n:m], f(b).cpu().double().numpy()[:, :, n:m].swapaxes(1, 2))
    assert np.isnan(c[:, m:]).all()


@pytest.mark.parametrize("m,n", [(20, 8), (300, 40)])
def test_zero_columns_give_identity_reflectors(m, n):
    """Columns whose subdiagonal part is zero (dlarfg's H = I, tau = 0), in
    the one-launch and the panel form, and through least squares."""
    A = np.zeros((1, m, n))
    A[0, :n] = np.triu(np.random.default_rng(1).standard_normal((n, n))) + 4 * np.eye(n)
    A[0, n:, 5] = 1.0
    h, tau0 = np.linalg.qr(A, mode="raw")
    t = torch.from_numpy(np.ascontiguousarray(np.swapaxes(A, 1, 2))).cuda()
    a = t.clone()
    tau = api.geqrf_batched(a).cpu().numpy()
    assert (tau[0, :5] == 0).all() and tau[0, 5] > 0
    assert np.max(np.abs(tau - tau0)) <= 1e-13
    assert np.max(np.abs(a.cpu().numpy() - h)) <= 1e-13 * np.abs(h).max()
    b = torch.ones(1, 1, m, dtype=torch.float64, device="cuda")
    api.gels_batched(t, b)
    ref = np.linalg.lstsq(A[0], np.ones(m), rcond=None)[0]
    assert np.max(np.abs(b.cpu().numpy()[0, 0, :n] - ref)) <= 1e-12 * np.abs(ref).max()


def test_more_right_hand_sides_than_one_launch_holds():
    m, n, nrhs, k = 40, 24, 300, 2
    r = np.random.default_rng(3)
    A, B = r.standard_normal((k, m, n)), r.standard_normal((k, m, nrhs))
    ta = torch.from_numpy(np.ascontiguousarray(np.swapaxes(A, 1, 2))).cuda()
    tb = torch.from_numpy(np.ascontiguousarray(np.swapaxes(B, 1, 2))).cuda()
    api.gels_batched(ta, tb)
    X = np.swapaxes(tb.cpu().numpy(), 1, 2)[:, :n]
    for i in range(k):
        ref = np.linalg.lstsq(A[i], B[i], rcond=None)[0]
        assert np.max(np.abs(X[i] - ref)) <= 1e-11 * np.abs(ref).max()


# Column 0 is (0, 1, .., 1): tau = 1 and v_i = 1 / sqrt(m - 1).  The last column
# is (1, e, .., e) with v_i e = 0.9 half ulps of 1, so R(0, n - 1) = -sqrt(m - 1) e
# exactly, formed as 1 - (1 + sum).  With the unit entry's product added last the
# sum rounds twice at size 1 (it, and the scaling by tau); terms summed onto the
# 1 one by one would all be lost.  Short and tall columns, and a panel's trailing one.
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("m,n", [(64, 2), (112, 8), (250, 8), (256, 40), (600, 40), (1024, 40)])
def test_unit_entry_joins_last(m, n, dtype):
    u = torch.finfo(dtype).eps / 2
    A = np.random.default_rng(m + n).standard_normal((m, n))
    e = float(torch.tensor(0.9 * u * np.sqrt(m - 1)).to(dtype))
    A[:, 0], A[:, n - 1] = 1.0, e
    A[0, 0], A[0, n - 1] = 0.0, 1.0
    tA = torch.from_numpy(np.ascontiguousarray(A.T)[None]).to(dtype).cuda()
    api.geqrf_batched(tA)
    got, want = float(tA[0, n - 1, 0]), np.sqrt(m - 1) * e
    assert abs(abs(got) - want) <= 2.05 * u + 4 * m * u * want
