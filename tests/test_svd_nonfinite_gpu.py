"""The SVD of matrices with NaN, infinite or overflowing entries: the call
returns, those matrices say so in their singular values, and their neighbours
in the batch get what they get without them, bit for bit (a workgroup works on
one matrix)."""
import pytest
import torch

from gputils_amd import api

pytestmark = pytest.mark.gpu

# in LDS, parked, G in the workspace, all in the workspace (more than 64 columns)
SHAPES = [(1, 1), (20, 10), (60, 30), (96, 64), (97, 40), (420, 60), (150, 70)]


@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("full", [True, False])
def test_neighbours(m, n, dtype, full):
    g = torch.Generator().manual_seed(100 * m + n)
    clean = torch.randn(8, n, m, generator=g, dtype=torch.float64).to(dtype)
    t = clean.clone()
    t[1, n // 2, m // 3] = float("nan")
    t[2, 0, 0] = float("inf")
    t[4, n - 1, m - 1] = float("-inf")
    t[5] = float("nan")
    t[6, n // 2] *= torch.finfo(dtype).max / 16  # finite, its square is not
    got = api.gesvd_batched(t.cuda(), compute_u=True, compute_v=full)
    want = api.gesvd_batched(clean.cuda(), compute_u=True, compute_v=full)
    torch.cuda.synchronize()
    for k in (0, 3, 7):
        for x, y in zip(got, want):
            if x is not None:
                assert torch.equal(x[k], y[k])
    S = got[0].cpu()
    for k in (1, 2, 4, 5):
        assert not bool(torch.isfinite(S[k]).all())
