"""Direct sums and energies on both sides of the line (1,024) up to which the
records are packed on the host.

One context takes small and large sets in turn, so that a set left from the
call before would show. Bounds as in the other direct sums' test: a term has a
relative error below 16 roundings, a sum of n terms one below n."""
import numpy as np
import pytest

from bhgpu import ic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(1, 2, 3, 255), (1023, 1024, 1025, 1024, 1), (2048, 1024, 2049, 2)])
def test_few_points(gpu, sizes):
    for turn, n in enumerate(sizes):
        p = ic.plummer(n, 20 + turn)
        print(f"few points n={n}", flush=True)
        x, m = p["pos"], p["mass"]
        idx = np.unique([0, n // 2, n - 1]).astype(np.uint32)
        for sel in (idx, None):
            got = gpu.direct_sum(p, sel, 1e-4)
            got = got if sel is not None else got[idx]
            for k, i in enumerate(idx):
                d = x - x[i]
                r2 = (d * d).sum(1) + 1e-4
                t = d * (m / (r2 * np.sqrt(r2)))[:, None]
                assert (np.abs(got[k] - t.sum(0)) <= (n + 16) * 2.0 ** -52 * np.abs(t).sum(0)).all()
        _, pot = gpu.energies(p)
        r = np.sqrt(((x[:, None] - x[None]) ** 2).sum(2))[np.triu_indices(n, 1)]
        pairs = (m[:, None] * m[None])[np.triu_indices(n, 1)] / r
        assert abs(pot + pairs.sum()) <= (n + 16) * 2.0 ** -52 * pairs.sum()
