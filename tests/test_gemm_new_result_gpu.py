"""gemm_batched without a given C takes uninitialised memory for it: every
entry is written, and none is read, on each of the product kernels."""
import numpy as np
import pytest
import torch

from gputils_amd import api

pytestmark = pytest.mark.gpu


# one shape per route, as in the test of the values: whole matrices in LDS, registers, a vector, odd shapes, tiles
@pytest.mark.parametrize("m,n,k", [(64, 64, 64), (128, 128, 128), (64, 1, 64), (5, 3, 7), (48, 40, 32), (100, 50, 75),
                                   (200, 17, 129)])
@pytest.mark.parametrize("dtype,mode", [(torch.float32, "fp32"), (torch.float32, "bf16x3"), (torch.float64, "fp32")])
def test_poisoned_memory(m, n, k, dtype, mode, monkeypatch):
    r = np.random.default_rng(m * n + k)
    A = torch.from_numpy(r.standard_normal((3, k, m))).to(dtype).cuda()
    B = torch.from_numpy(r.standard_normal((3, n, k))).to(dtype).cuda()
    want = api.gemm_batched(A, B, torch.zeros(3, n, m, dtype=dtype, device="cuda"), mode=mode)
    monkeypatch.setattr(api.torch, "empty", lambda *a, **kw: torch.full(*a, float("nan"), **kw))
    assert torch.equal(api.gemm_batched(A, B, mode=mode), want)
