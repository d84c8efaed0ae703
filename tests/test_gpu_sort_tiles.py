"""Radix passes at the edges of their tiles: 2,048 keys up to 262,144 particles,
4,096 above. Keys, order and nodes equal the oracle's bit for bit; a batch of
the same total equals its systems alone."""
import numpy as np
import pytest

from bhgpu import ic, layout

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [14335, 14336, 14337, 262143, 262144, 262145])
def test_tile_edges(gpu, orc, n):
    p = ic.hernquist(n, 9)
    print(f"tiles n={n}", flush=True)
    gpu.build_tree(p, 64, 256)
    ge, oe = gpu.export(), orc.build(p, 64, 256).export()
    for k in ("keys", "perm", "particles", "nodes", "groups"):
        assert ge[k].tobytes() == oe[k].tobytes(), k


@pytest.mark.parametrize("sizes", [[2048, 1, 2047, 100000, 160049], [160049, 100000, 2047, 1, 2048]])
def test_tile_edges_batch(gpu, sizes):
    fp = layout.force_params(0.9, 1e-4, 1.0, False)
    parts = [ic.plummer(n, 3) if n > 1 else ic.random_box(1, 3, 1.0) for n in sizes]
    table = np.concatenate([layout.system(len(q), fp, 32, 64, 32, 1e-3, 1e-3) for q in parts])
    print(f"tiles batch of {sum(sizes)}", flush=True)
    out, _ = gpu.step_batch(np.concatenate(parts), table)
    lo = 0
    for q in parts:
        assert out[lo:lo + len(q)].tobytes() == gpu.step(q, fp, 32, 64, 32, 1e-3, 1e-3)[0].tobytes(), len(q)
        lo += len(q)
