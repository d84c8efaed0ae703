"""The sort's runs of equal leading key bits.

The radix passes order keys by their leading 32, 40 or 48 bits; runs of equal
leading bits are ordered by the bits below them in registers (up to 64 keys),
in memory (up to 1,024) or, longer, by a second attempt with full keys. A far
outlier widens the domain so that everything else shares leading bits. Keys,
permutation and nodes equal the oracle's bit for bit, for one system and for
systems of a batch alone and together."""
import numpy as np
import pytest

from bhgpu import ic, layout
from bhgpu import lib as bl

pytestmark = pytest.mark.gpu


def clump(n, seed, far, dup=0):
    """n particles in a unit box, the last one at distance far; dup of them at one place."""
    p = ic.random_box(n, seed, 1.0)
    if dup:
        p["pos"][5:5 + dup] = p["pos"][3]
    p["pos"][-1] = far
    return p


# far: the box spans 2^-18 .. 2^-9 of the domain, so the leading levels split
# it into nothing, a few cells or many; n on both sides of the pass rule
CASES = [(2, 2.0 ** 17, 0), (60, 2.0 ** 18, 0), (65, 2.0 ** 17, 0), (1000, 2.0 ** 16, 30), (1025, 2.0 ** 18, 0),
         (3000, 2.0 ** 10, 200), (5000, 2.0 ** 17, 3000), (32768, 2.0 ** 9, 1500), (33000, 2.0 ** 12, 0),
         (40000, 2.0 ** 15, 500)]


@pytest.mark.parametrize("n,far,dup", CASES)
def test_runs_of_equal_leading_bits(orc, n, far, dup):
    p = clump(n, 17, far, dup)
    print(f"runs n={n} far={far} dup={dup}", flush=True)
    with bl.Context(0) as gpu:  # of its own: a context whose runs were too long keeps to full keys
        gpu.build_tree(p, 8, 64)
        ge = gpu.export()
    oe = orc.build(p, 8, 64).export()
    for k in ("keys", "perm", "particles", "nodes", "center", "iab", "groups"):
        assert ge[k].tobytes() == oe[k].tobytes(), k


@pytest.mark.parametrize("cases", [CASES, [c for c in CASES if c[0] < 1025 or c[1] < 2.0 ** 14]])
def test_runs_end_at_systems(cases):
    fp = layout.force_params(0.5, 1e-4, 1.0, True)
    parts = [clump(n, 40 + i, far, dup) for i, (n, far, dup) in enumerate(cases)]
    table = np.concatenate([layout.system(len(q), fp, 8, 64, 32, 1e-3, 1e-3) for q in parts])
    print(f"batch of {len(parts)}", flush=True)
    with bl.Context(0) as gpu:
        out, _ = gpu.step_batch(np.concatenate(parts), table)
        lo = 0
        for q in parts:
            alone, _ = gpu.step(q, fp, 8, 64, 32, 1e-3, 1e-3)
            assert out[lo:lo + len(q)].tobytes() == alone.tobytes(), len(q)
            lo += len(q)
