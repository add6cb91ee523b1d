"""Short reductions (one launch) of vectors with infinities, NaNs, zeros and
subnormal numbers, against a model of the two launches that longer vectors
take: the partition, the order of combination (which decides whether a maximum
past a NaN shows) and the rescaling of the norm.  The entries are small
integers, so sums are exact in any order and results agree exactly."""
import numpy as np
import pytest
import torch

from gputils_amd import api

pytestmark = pytest.mark.gpu


def combine(op, a, b):
    with np.errstate(invalid="ignore"):
        if op == "amax":
            return np.where(a > b, a, b)
        if op == "amin":
            return np.where(a < b, a, b)
        return a + b


def block(op, v):
    """v (groups, 256): 64-lane butterflies, then the four wavefronts in turn."""
    w = v.reshape(v.shape[0], 4, 64)
    for off in (32, 16, 8, 4, 2, 1):
        o = w[:, :, np.arange(64) ^ off]
        with np.errstate(invalid="ignore"):
            w = np.where(o > w, o, w) if op == "amax" else np.where(o < w, o, w) if op == "amin" else w + o
    r = w[:, 0, 0]
    for k in range(1, 4):
        r = combine(op, r, w[:, k, 0])
    return r


def total(op, e):
    """Two passes: workgroups of 256 threads over eight entries a thread, then one over their partials."""
    identity = np.inf if op == "amin" else 0.0
    groups = -(-len(e) // 2048)
    acc = np.full(groups * 256, identity)
    for i in range(0, len(e), groups * 256):
        part = e[i:i + groups * 256]
        acc[:len(part)] = combine(op, acc[:len(part)], part)
    partial = np.full(256, identity)
    partial[:groups] = combine(op, partial[:groups], block(op, acc.reshape(groups, 256)))
    return block(op, partial[None])[0]


def model(fn, x, dtype):
    with np.errstate(all="ignore"):
        if fn == "dot":
            r = total(fn, x * np.ones_like(x))
        elif fn == "nrm2":
            r = np.sqrt(total("sum", x * x))
            a = np.abs(x)
            big = np.max(a[~np.isnan(a)], initial=0.0)
            if big > 0 and (big > 1e140 or big < 1e-140):
                r = big * np.sqrt(total("sum", (x * (1.0 / big)) ** 2))
        else:
            r = total(fn, np.where(x < 0, -x, x))
        return float(np.asarray(r).astype(np.float32 if dtype == torch.float32 else np.float64))


def vectors(n, dtype):
    r = np.random.default_rng(n)
    x = r.integers(1, 9, n).astype(float) * r.choice([-1.0, 1.0], n)
    for at in sorted({0, n // 3, n // 2, n - 1}):
        for v in (np.inf, -np.inf, np.nan, 0.0):
            y = x.copy()
            y[at] = v
            yield f"{v} at {at}", y
    if n > 1:
        y = x.copy()
        y[0], y[n - 1] = np.inf, np.nan
        yield "both", y
    yield "zeros", np.zeros(n)
    yield "subnormal", np.full(n, 2.0 ** -149 if dtype == torch.float32 else 2.0 ** -1074)


@pytest.mark.parametrize("n", [1, 65, 2048, 2049, 6145, 8192])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_as_two_launches(n, dtype):
    ones = torch.ones(n, dtype=dtype, device="cuda")
    for name, x in vectors(n, dtype):
        tx = torch.from_numpy(x).to(dtype).cuda()
        for fn in ("dot", "nrm2", "asum", "amax", "amin"):
            got = float(api.dot(tx, ones) if fn == "dot" else getattr(api, fn)(tx))
            want = model(fn, x, dtype)
            assert got == want or (np.isnan(got) and np.isnan(want)), (name, fn, got, want)
