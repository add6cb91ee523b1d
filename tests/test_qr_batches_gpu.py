"""QR, least squares and Q application of batches: 130 tall matrices at the
rows where the kernels change and around multiples of a panel's columns, and
ormqr with four columns a wavefront.

Two different matrices, repeated over the batch; every copy has to come out
the same, and the two agree with numpy in 64 bits (Gaussian, m >= 1.3 n, so to
20 n eps: 1e-11 in FP64, 20 * 160 * 6e-8 = 2e-4 in FP32)."""
import numpy as np
import pytest
import torch

from gputils_amd import api

pytestmark = pytest.mark.gpu

BATCH = 130


def tol(dtype):
    return 1e-11 if dtype == torch.float64 else 2e-4


def put(M, dtype, batch):
    """(2, m, n) -> (batch, n, m) storage, the two in turn."""
    t = torch.from_numpy(np.ascontiguousarray(np.swapaxes(M, 1, 2))).to(dtype).cuda()
    return t.repeat((batch + 1) // 2, 1, 1)[:batch].contiguous()


def two(t):
    """The two results, after every other copy has been compared with its own."""
    assert torch.equal(t[::2], t[:1].expand_as(t[::2])) and torch.equal(t[1::2], t[1:2].expand_as(t[1::2]))
    return t[:2].double().cpu().numpy()


def limits():
    for dtype, widths in ((torch.float64, (80, 48, 16)), (torch.float32, (160, 96, 64))):
        for ms, w in (((257, 384), widths[0]), ((385, 640), widths[1]), ((641, 1024), widths[2])):
            for m in ms:
                for n in (w, w + 1):
                    yield pytest.param(m, n, dtype, id=f"{m}x{n}-{'d' if dtype == torch.float64 else 's'}")


@pytest.mark.parametrize("m,n,dtype", limits())
def test_tall_batches(m, n, dtype):
    r = np.random.default_rng(m + n)
    A, B = r.standard_normal((2, m, n)), r.standard_normal((2, m, 3))
    h, tau0 = np.linalg.qr(A, mode="raw")
    t = put(A, dtype, BATCH)
    tau = api.geqrf_batched(t)
    assert np.abs(two(t) - h).max() <= tol(dtype) * np.abs(h).max()
    assert np.abs(two(tau[:, None])[:, 0] - tau0).max() <= 2 * tol(dtype)
    # least squares whose columns and right-hand sides together are n
    a, b = put(A[:, :, :n - 3], dtype, BATCH), put(B, dtype, BATCH)
    was = b.clone()
    api.gels_batched(a, b)
    X = np.swapaxes(two(b), 1, 2)
    for i in range(2):
        ref = np.linalg.lstsq(A[i][:, :n - 3], B[i], rcond=None)[0]
        assert np.abs(X[i][:n - 3] - ref).max() <= tol(dtype) * np.abs(ref).max()
    assert torch.equal(b[:, :, n - 3:], was[:, :, n - 3:])


@pytest.mark.parametrize("m,n", [(257, 17), (300, 40), (1000, 33)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_results_do_not_depend_on_the_batch(m, n, dtype):
    """Factors and solutions of the first matrices of 200, and of these alone: bit for bit."""
    r = np.random.default_rng(m * n)
    A, B = (torch.from_numpy(r.standard_normal(s)).to(dtype).cuda() for s in ((200, n, m), (200, 2, m)))
    for k in (1, 100):
        for fn in (lambda a, b: api.geqrf_batched(a), api.gels_batched):
            a, b, a1, b1 = A.clone(), B.clone(), A[:k].clone(), B[:k].clone()
            fn(a, b)
            fn(a1, b1)
            assert torch.equal(a[:k], a1) and torch.equal(b[:k], b1)


# one to ten registers a column; more than 64 reflectors where there are rows for them
@pytest.mark.parametrize("m,k", [(64, 64), (128, 75), (256, 150), (384, 70), (640, 131), (641, 66)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_four_columns_a_wavefront(m, k, dtype):
    ncols, batch = 131, 126  # 16506 columns; the last wavefront of a matrix holds three
    r = np.random.default_rng(m + k)
    A, C = r.standard_normal((2, m, k)), r.standard_normal((2, m, ncols))
    t, c = put(A, dtype, batch), put(C, dtype, batch)
    tau = api.geqrf_batched(t)
    Q, _ = np.linalg.qr(A, mode="complete")
    if k == m:  # numpy's last reflector is the identity, and so is geqrf's
        assert (two(tau[:, None])[:, 0, -1] == 0).all()
    for trans in (True, False):
        got = np.swapaxes(two(api.ormqr_batched(t, tau, c.clone(), trans=trans)), 1, 2)
        want = (np.swapaxes(Q, 1, 2) if trans else Q) @ C
        assert np.abs(got - want).max() <= tol(dtype) * np.abs(want).max()
