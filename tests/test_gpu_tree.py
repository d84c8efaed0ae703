"""Tree construction at the edges of its tiles and levels, bit for bit against the oracle.

Depths from 0 up put the nodes of a single system's upper levels, which one
workgroup finishes, at none, some or all of the tree's; sizes lie around the
tile of 4,096 particles and the 1,024 threads that share it."""
import pytest

from bhgpu import ic, layout

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ml", [(1, 1), (2, 1), (3, 64), (9, 8), (65, 8), (129, 128), (513, 1), (1023, 4), (1025, 64),
                                  (4095, 2), (4096, 32), (4097, 128), (8193, 1), (12289, 16)])
def test_tree_edges(gpu, orc, n, ml):
    for p in (ic.random_box(n, 7, 1.0), ic.plummer(n, 8)):
        print(f"tree n={n} ml={ml}", flush=True)
        gpu.build_tree(p, ml, 256)
        ge, oe = gpu.export(), orc.build(p, ml, 256).export()
        for k in ("keys", "perm", "particles", "nodes", "center", "iab", "groups"):
            assert ge[k].tobytes() == oe[k].tobytes(), k
