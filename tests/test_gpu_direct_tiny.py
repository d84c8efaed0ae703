"""Direct sums over particles closer together than the root of the smallest double.

The square of such a distance is zero or has few digits left, while the distance
itself is not zero: without softening the pull is infinite, as a sum of plain
square roots and divisions has it, and only of coinciding coordinates not a
number. Bounds of finite sums as in the other direct sums' test."""
import numpy as np
import pytest

from bhgpu import ic

pytestmark = pytest.mark.gpu


def reference(p, idx, eps2):
    x, m = p["pos"], p["mass"]
    acc, size = np.zeros((len(idx), 3)), np.zeros((len(idx), 3))
    with np.errstate(all="ignore"):
        for k, i in enumerate(idx):
            d = np.delete(x, i, 0) - x[i]
            r2 = (d * d).sum(1) + eps2
            t = d * (np.delete(m, i) * (1.0 / (r2 * np.sqrt(r2))))[:, None]
            acc[k], size[k] = t.sum(0), np.abs(t).sum(0)
    return acc, size


@pytest.mark.parametrize("n", [2, 3, 257, 700])
@pytest.mark.parametrize("eps2", [0.0, 1e-4])
@pytest.mark.parametrize("apart", [1e-300, 1e-170, 1e-158, 1e-140, 1e-100])
@pytest.mark.parametrize("zero", [False, True])
def test_tiny_distances(gpu, n, eps2, apart, zero):
    # two of them (one at zero itself, or on either side of it), the last ones,
    # so that with 257 only one is in the second tile
    p = ic.plummer(n, 3)
    p["pos"][n - 2] = 0.0 if zero else -2 * apart
    p["pos"][n - 1] = (apart, 2 * apart, 3 * apart)
    idx = np.unique([0, n - 2, n - 1]).astype(np.uint32)
    print(f"direct tiny n={n} eps2={eps2} apart={apart} zero={zero}", flush=True)
    ref, size = reference(p, idx, eps2)
    for sel in (idx, None):
        got = gpu.direct_sum(p, sel, eps2)
        got = got if sel is not None else got[idx]
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        ok = np.isfinite(ref)
        assert np.array_equal(got[~ok], ref[~ok], equal_nan=True)
        assert (np.abs(got[ok] - ref[ok]) <= ((n + 16) * 2.0 ** -52 * size)[ok]).all()
