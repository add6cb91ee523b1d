"""Several threads, each on its own stream, with sizes of one kernel that need
different amounts of dynamic LDS: every call is accepted and right."""
import threading

import pytest
import torch

from gputils_amd import api

pytestmark = pytest.mark.gpu


def test_solves_of_different_sizes_at_once():
    jobs = {}
    for n in (400, 440, 480, 512, 520, 600, 672):
        g = torch.Generator(device="cuda").manual_seed(n)
        M = torch.randn(2, n, n, generator=g, device="cuda", dtype=torch.float64)
        A = (M @ M.transpose(1, 2).contiguous() / n + 2 * torch.eye(n, device="cuda", dtype=torch.float64)).contiguous()
        B = torch.randn(2, 1, n, generator=g, device="cuda", dtype=torch.float64)
        L = A.clone()
        api.potrf_batched(L)
        jobs[n] = (L, B, _solve(L, B))
    torch.cuda.synchronize()
    errors = []

    def work(n):
        try:
            L, B, want = jobs[n]
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(40):
                    got = _solve(L, B)
                torch.cuda.current_stream().synchronize()
                assert torch.equal(got, want)
        except Exception as e:  # noqa: BLE001
            errors.append((n, e))

    threads = [threading.Thread(target=work, args=(n,)) for n in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def _solve(L, B):
    X = B.clone()
    api.potrs_batched(L, X)
    return X
