"""Staging memory that passes from one request of a server to the next.

Requests of equal, smaller and larger sizes follow each other through the same
server, refused ones among them (each double of a record not finite in turn);
every result is that of the request stepped alone, bit for bit."""
import numpy as np
import pytest

from bhgpu import ic, layout
from bhgpu import lib as bl

pytestmark = pytest.mark.gpu


def test_staging_reuse(gpu):
    srv = bl.Server(gpu)
    fp = layout.force_params(0.5, 1e-4, 1.0, True)
    fields = [("mass", None)] + [(f, a) for f in ("pos", "vel") for a in range(3)]
    for turn, sizes in enumerate([(1, 300, 257, 4000), (300, 1, 4000, 255), (4100, 150, 3999, 2, 4000)]):
        specs = {}
        for k, n in enumerate(sizes):
            p = ic.plummer(n, 10 * turn + k)
            bad = p.copy()
            f, a = fields[(7 * turn + k) % len(fields)]
            bad[f][(n - 1,) if a is None else (n - 1, a)] = (np.nan, np.inf, -np.inf)[k % 3]
            with pytest.raises(bl.BHError):
                srv.submit(bad, bl.request(n, 0.5, 1e-4, steps=1, max_leaf=16))
            specs[srv.submit(p, bl.request(n, 0.5, 1e-4, steps=1, max_leaf=16, target_size=32))] = p
        got = {}
        while srv.pending() != (0, 0):
            srv.step()
            got.update((t, r) for t, r, _ in srv.poll())
        for t, p in specs.items():
            print(f"turn {turn} n={len(p)}", flush=True)
            for kick, drift in ((5e-4, 1e-3), (5e-4, 0.0)):
                p, _ = gpu.step(p, fp, 16, 256, 32, kick, drift)
            assert got[t].tobytes() == p.tobytes()
    srv.close()
