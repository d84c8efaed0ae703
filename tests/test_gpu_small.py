"""Small systems, whose particles a few workgroups order.

Blocks of 1,024 are sorted by 54 leading key bits and the index, their runs of
equal bits by the rest of the key, and merged. Sizes at the edges of blocks and
of the range, with a far particle that squeezes the others into a few cells and
many at one place, in every block: keys, order, particles and nodes equal the
oracle's bit for bit. Resident steps, which build from compact positions, equal
steps on records."""
import numpy as np
import pytest

from bhgpu import ic, layout
from bhgpu import lib as bl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 1023, 1024, 1025, 2048, 3000, 4096, 5119, 11265, 12287, 12288, 12289])
@pytest.mark.parametrize("far,same", [(0.0, 0), (2.0 ** 12, 0), (2.0 ** 19, 0), (2.0 ** 16, 3), (0.0, 1)])
def test_small_sort(gpu, orc, n, far, same):
    p = ic.random_box(n, 3 + n, 1.0)
    if same:
        p["pos"][:: same] = p["pos"][0]  # 1: all of them
    if far:
        p["pos"][n // 2] = (far, -far, 1.0)
    print(f"small n={n} far={far} same={same}", flush=True)
    gpu.build_tree(p, 16, 64)
    ge, oe = gpu.export(), orc.build(p, 16, 64).export()
    for k in ("keys", "perm", "particles", "nodes", "center", "iab", "groups"):
        assert ge[k].tobytes() == oe[k].tobytes(), k


@pytest.mark.parametrize("n", [700, 1025, 12288])
def test_small_resident_steps(n):
    fp = layout.force_params(0.6, 1e-4, 1.0, True)
    with bl.Context(0) as one, bl.Context(0) as two:
        p = ic.plummer(n, 6)
        one.state_upload(p)
        for k in range(4):
            print(f"resident n={n} step {k}", flush=True)
            one.state_step(fp, 8, 256, 32, 1e-3, 1e-3)
            p, _ = two.step(p, fp, 8, 256, 32, 1e-3, 1e-3)
            assert one.state_download().tobytes() == p.tobytes()
