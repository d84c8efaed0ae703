"""The direct sum's tiles of 256 sources, its own-source check and its two forms.

Sources and targets whose distances stay finite go through the reciprocal
square root, others (any coordinate of 1e150 or more, or not a number) through
the square root and the division. Both against the sum in numpy's float64:
a term of either has a relative error below 16 roundings and a sum of n terms
one below n, so an acceleration is within (n + 16) 2^-52 of the sum of its
terms' magnitudes."""
import numpy as np
import pytest

from bhgpu import ic

pytestmark = pytest.mark.gpu


def reference(p, idx, eps2):
    x, m = p["pos"].astype(np.float64), p["mass"].astype(np.float64)
    acc, size = np.zeros((len(idx), 3)), np.zeros((len(idx), 3))
    with np.errstate(all="ignore"):
        for k, i in enumerate(idx):
            d = np.delete(x, i, 0) - x[i]
            r2 = (d * d).sum(1) + eps2
            t = d * (np.delete(m, i) * (1.0 / (r2 * np.sqrt(r2))))[:, None]
            acc[k], size[k] = t.sum(0), np.abs(t).sum(0)
    return acc, size


@pytest.mark.parametrize("n,eps2", [(1, 1e-4), (2, 0.0), (255, 1e-6), (256, 0.0), (257, 1e-4), (513, 1e300), (1500, 1e-250)])
@pytest.mark.parametrize("wild", ["none", "far", "infinite", "nan", "heavy", "twins"])
def test_direct_forms(gpu, n, eps2, wild):
    p = ic.plummer(n, 3)
    j = n // 2
    if wild == "far":
        p["pos"][j] = (1e160, -2e151, 0.0)
    elif wild == "infinite":
        p["pos"][j, 1] = np.inf
    elif wild == "nan":
        p["pos"][j, 2] = np.nan
    elif wild == "heavy":
        p["mass"][j] = np.inf
    elif wild == "twins":  # without softening their pull is not a number
        p["pos"][j] = p["pos"][0]
    idx = np.unique([0, j, n - 1, n // 3, min(n - 1, 255), min(n - 1, 256)]).astype(np.uint32)
    print(f"direct n={n} eps2={eps2} {wild}", flush=True)
    for sel in (idx, None):
        got = gpu.direct_sum(p, sel, eps2)
        got = got if sel is not None else got[idx]
        ref, size = reference(p, idx, eps2)
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        ok = np.isfinite(ref) & np.isfinite(size)
        assert np.array_equal(got[~ok & ~np.isnan(ref)], ref[~ok & ~np.isnan(ref)])
        assert (np.abs(got - ref)[ok] <= ((n + 16) * 2.0 ** -52 * size)[ok]).all()


def test_records_loaded_in_pieces(gpu):
    """Records go to the GPU 2^20 at a time; the last piece holds three."""
    n = (1 << 20) + 3
    p = ic.uniform_cube(n, 4)
    idx = np.array([0, (1 << 20) - 1, 1 << 20, n - 1], np.uint32)
    print(f"direct n={n}", flush=True)
    ref, size = reference(p, idx, 1e-6)
    assert (np.abs(gpu.direct_sum(p, idx, 1e-6) - ref) <= (n + 16) * 2.0 ** -52 * size).all()


@pytest.mark.parametrize("n,m", [(1 << 19, 1), ((1 << 19) + 3, 7), ((1 << 19) + 3, 4096), ((1 << 19) + 3, 4097), ((1 << 20) + 3, 8193)])
@pytest.mark.parametrize("wild", ["none", "far", "nan"])
def test_sources_summed_as_they_arrive(gpu, n, m, wild):
    """Up to n / 128 targets of at least 2^19 particles are summed piece by
    piece of 2^18 sources; beside that line all sources come first."""
    p = ic.uniform_cube(n, 5)
    last = n - 1 if wild == "far" else n - 2
    if wild == "far":  # in the last piece
        p["pos"][last] = (1e160, -2e151, 0.0)
    elif wild == "nan":
        p["mass"][last] = np.nan
    edges = [0, (1 << 18) - 1, 1 << 18, (1 << 19) - 1, n - 1, n - 1, n // 3]
    idx = np.array((edges * (m // len(edges) + 1))[:m], np.uint32)
    print(f"direct n={n} m={m} {wild}", flush=True)
    got = gpu.direct_sum(p, idx, 1e-6)
    first = min(m, len(edges))
    ref, size = reference(p, idx[:first], 1e-6)
    assert np.array_equal(np.isnan(got[:first]), np.isnan(ref))
    ok = np.isfinite(ref)
    assert (np.abs(got[:first] - ref)[ok] <= ((n + 16) * 2.0 ** -52 * size)[ok]).all()
    for k in range(first, m, 997):  # the same target is the same sum
        assert np.array_equal(got[k], got[k % len(edges)], equal_nan=True)


@pytest.mark.parametrize("n", [2, 3, 63, 64, 65, 127, 128, 129, 500, 1025, 4001, 10001, 16384, 16385, 24576, 24577])
def test_pair_grids(gpu, n):
    """The grids of pair sums at sizes where the number of windows changes: the
    potential energy against numpy's float64 sum and its error bound of n
    roundings of a sum of terms of one sign, and all targets' accelerations."""
    p = ic.plummer(n, 7)
    x, m = p["pos"], p["mass"]
    pot = 0.0
    for i in range(n - 1):
        d = x[i + 1:] - x[i]
        pot -= m[i] * (m[i + 1:] / np.sqrt((d * d).sum(1))).sum()
    print(f"pairs n={n}", flush=True)
    _, got = gpu.energies(p)
    assert abs(got - pot) <= (n + 16) * 2.0 ** -52 * abs(pot)
    idx = np.unique([0, n // 2, n - 1])
    ref, size = reference(p, idx, 1e-4)
    assert (np.abs(gpu.direct_sum(p, None, 1e-4)[idx] - ref) <= (n + 16) * 2.0 ** -52 * size).all()
