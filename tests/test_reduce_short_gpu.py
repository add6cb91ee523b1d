"""Reductions of short vectors: the single launch and its edges."""
import numpy as np
import pytest
import torch

from gputils_amd import api

pytestmark = pytest.mark.gpu


# one group, its edges, two to four groups with remainders, the last single launch
@pytest.mark.parametrize("n", [1, 63, 65, 2047, 2048, 2049, 4097, 6145, 8191, 8192, 8193])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_short_reductions(n, dtype):
    r = np.random.default_rng(n)
    tx = torch.from_numpy(r.standard_normal(n)).to(dtype).cuda()
    ty = torch.from_numpy(r.standard_normal(n)).to(dtype).cuda()
    x, y = tx.double().cpu().numpy(), ty.double().cpu().numpy()
    # FP64 accumulation, then one rounding to the result's type
    eps = torch.finfo(dtype).eps
    tol = eps + n * 2.3e-16
    assert abs(float(api.dot(tx, ty)) - x @ y) <= tol * (np.abs(x) @ np.abs(y))
    assert np.isclose(float(api.nrm2(tx)), np.linalg.norm(x), rtol=tol, atol=0)
    assert np.isclose(float(api.asum(tx)), np.abs(x).sum(), rtol=tol, atol=0)
    assert float(api.amax(tx)) == np.abs(x).max()
    assert float(api.amin(tx)) == np.abs(x).min()


@pytest.mark.parametrize("n", [257, 8192])
@pytest.mark.parametrize("scale", [1e-200, 1e200])
def test_short_nrm2_rescaled(n, scale):
    x = np.random.default_rng(n).standard_normal(n)
    got = float(api.nrm2(torch.from_numpy(x * scale).cuda()))
    assert np.isclose(got, np.linalg.norm(x) * scale, rtol=n * 2.3e-16 + 1e-15, atol=0)
