"""The general product kernel at its edges: tiles of 32 and 64 with one row or
column more or less, chunks of 16 and 32 in k with remainders, the empty
product, alpha and beta, padded operands.  The padding of A and B holds NaN
(never used) and so does C's, which stays; C is NaN where beta = 0.

Against 64 bits, entries in [-1, 1]: |error| <= (k + 2) u sum_p |a_ip b_pj| for
FP32 and FP64; the split-BF16 products drop the al bl term and round each
term's remainder, 2^-16 per product and 2^-15 with margin for the FP32 sums."""
import ctypes

import numpy as np
import pytest
import torch

from gputils_amd import api
from gputils_amd._lib import lib

pytestmark = pytest.mark.gpu

SHAPES = [(5, 6, 0), (7, 9, 1), (32, 32, 15), (31, 17, 33), (16, 31, 17), (33, 32, 16), (32, 33, 20), (48, 49, 31),
          (64, 63, 47), (65, 64, 65), (96, 97, 32), (100, 75, 50), (129, 80, 100), (81, 144, 3)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("mode", ["fp32", "bf16x3", "fp64"])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (-1.5, 0.5)])
def test_padded_products(m, n, k, mode, alpha, beta):
    batch, lda, ldb, ldc = 3, m + 1, max(k, 1) + 3, m + 5
    r = np.random.default_rng(1000 * m + 10 * n + k)
    dt = torch.float64 if mode == "fp64" else torch.float32
    f = lambda x: torch.from_numpy(x).to(dt).cuda()  # noqa: E731
    A, B, C = (r.uniform(-1, 1, s) for s in ((batch, k, m), (batch, n, k), (batch, n, m)))
    a, b, c = np.full((batch, max(k, 1), lda), np.nan), np.full((batch, n, ldb), np.nan), np.full((batch, n, ldc), np.nan)
    a[:, :k, :m], b[:, :, :k] = A, B
    if beta != 0.0:
        c[:, :, :m] = C
    ta, tb, tc = f(a), f(b), f(c)
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    st = api.stream_handle()
    args = (m, n, k, alpha, P(ta), lda, lda * max(k, 1), P(tb), ldb, ldb * n, beta, P(tc), ldc, ldc * n, batch)
    if mode == "fp64":
        assert lib().gputils_dgemm_strided_batched(*args, st) == 0
    else:
        assert lib().gputils_sgemm_strided_batched(*args, 1 if mode == "bf16x3" else 0, st) == 0
    got = tc.cpu().double().numpy()
    At, Bt = ta.cpu().double().numpy()[:, :k, :m], tb.cpu().double().numpy()[:, :, :k]
    C0 = tc.new_tensor(C).cpu().double().numpy() if beta != 0.0 else np.zeros_like(C)
    ref = alpha * np.matmul(Bt, At) + beta * C0
    size = abs(alpha) * np.matmul(np.abs(Bt), np.abs(At)) + abs(beta) * np.abs(C0)
    u = {"fp32": 2.0 ** -24, "fp64": 2.0 ** -53, "bf16x3": 2.0 ** -24}[mode]
    tol = (k + 2) * u + (2.0 ** -15 if mode == "bf16x3" else 0.0)
    assert np.all(np.abs(got[:, :, :m] - ref) <= tol * size + 1e-300)
    assert np.isnan(got[:, :, m:]).all()


# one shape per route: whole matrices in LDS, registers, a vector, small odd shapes, tiles
@pytest.mark.parametrize("m,n,k", [(64, 64, 64), (128, 128, 128), (64, 1, 64), (5, 3, 7), (100, 50, 75), (200, 17, 129)])
@pytest.mark.parametrize("dtype,mode", [(torch.float32, "fp32"), (torch.float32, "bf16x3"), (torch.float64, "fp32")])
def test_new_result_is_written_whole(m, n, k, dtype, mode):
    r = np.random.default_rng(m * n + k)
    A = torch.from_numpy(r.standard_normal((3, k, m))).to(dtype).cuda()
    B = torch.from_numpy(r.standard_normal((3, n, k))).to(dtype).cuda()
    want = api.gemm_batched(A, B, torch.zeros(3, n, m, dtype=dtype, device="cuda"), mode=mode)
    old = torch.full((3, n, m), float("nan"), dtype=dtype, device="cuda")
    del old  # the allocator hands this block to the next result of its size
    assert torch.equal(api.gemm_batched(A, B, mode=mode), want)
