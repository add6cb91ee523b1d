"""The SVD at the edges of its register QR (96 | 97 rows, 64 | 65 rows with 32
| 33 columns) and of its Jacobi pairs (16, 32, 40, 48, 56, 64 columns and one
more): A = U S V^T, orthogonal factors, numpy's singular values.

All arithmetic ends in FP64: n eps times a few tens, 1e-12 of the largest
singular value; FP32 results are rounded once, so 64 such terms of a product
differ by at most 64 * 6e-8 < 1e-5."""
import numpy as np
import pytest
import torch

from gputils_amd import api

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (20, 16), (20, 17), (64, 32), (64, 33), (65, 32), (70, 40), (70, 41), (96, 48), (97, 48), (96, 49),
          (96, 56), (96, 57), (96, 64), (97, 64), (70, 65)]


@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_decomposition(m, n, dtype):
    k, tol = 3, 1e-12 if dtype == torch.float64 else 1e-5
    t = torch.from_numpy(np.random.default_rng(100 * m + n).standard_normal((k, n, m))).to(dtype).cuda()
    A = np.swapaxes(t.double().cpu().numpy(), 1, 2)
    S0 = np.linalg.svd(A, compute_uv=False)
    big = S0[:, :1]
    for full in (True, False):  # without V the sweeps run on the transposed triangle, in FP32 first for FP32
        S, U, VT, info = api.gesvd_batched(t, compute_u=True, compute_v=full)
        assert info.cpu().tolist() == [0] * k
        s = S.double().cpu().numpy()[:, 0]
        assert np.all(np.abs(s - S0) <= tol * big)
        u = api.to_matrices(U).double().cpu().numpy()
        assert np.abs(np.swapaxes(u, 1, 2) @ u - np.eye(m)).max() <= tol
        # u_j^T A has norm s_j, and the rest of U is orthogonal to A
        c = np.swapaxes(u, 1, 2) @ A
        assert np.all(np.abs(np.linalg.norm(c, axis=2)[:, :n] - S0) <= tol * big)
        assert np.abs(c[:, n:]).max(initial=0) <= tol * big.max()
        if full:
            vt = api.to_matrices(VT).double().cpu().numpy()
            assert np.abs(u[:, :, :n] * s[:, None] @ vt - A).max() <= tol * big.max()
            assert np.abs(vt @ np.swapaxes(vt, 1, 2) - np.eye(n)).max() <= tol
