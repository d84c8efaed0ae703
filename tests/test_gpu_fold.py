"""How long the FP32 walk sums in FP32 before it adds to an FP64 sum.

Targets of 33 to 128 particles of small systems are walked in pieces of up to
32, whose sums must not get longer than those of the whole targets. The
bounds are the median errors (of an acceleration, against the FP64 walk over the
same lists, geometric mean over systems) when they were walked whole."""
import numpy as np
import pytest

from bhgpu import ic, layout
from bhgpu import lib as bl

pytestmark = pytest.mark.gpu

WHOLE = {("plummer", 1000, 32, 96, 0.5): 6.41e-8, ("plummer", 1000, 16, 128, 0.6): 6.93e-8,
         ("plummer", 4096, 32, 96, 0.5): 5.69e-8, ("plummer", 4096, 16, 128, 0.6): 6.05e-8,
         ("box", 4096, 32, 96, 0.5): 7.53e-8, ("box", 4096, 16, 128, 0.6): 8.05e-8}


@pytest.mark.parametrize("case", list(WHOLE))
def test_sums_of_pieces_are_no_less_exact(gpu, case):
    kind, n, leaf, target, theta = case
    fp = layout.force_params(theta, 1e-4, 1.0, True)
    log = []
    print("fold", case, flush=True)
    try:
        for seed in range(100, 124 if n == 1000 else 112):
            p = ic.plummer(n, seed) if kind == "plummer" else ic.random_box(n, seed, 1.0)
            acc = {}
            for precision in (bl.BH_FP32, bl.BH_FP64):
                gpu.set_precision(precision)
                gpu.build_tree(p, leaf, 256)
                acc[precision], npp, npc, _ = gpu.accel(fp, target)
            off = np.linalg.norm(acc[bl.BH_FP32] - acc[bl.BH_FP64], axis=1)
            log.append(np.log(np.median(off / np.linalg.norm(acc[bl.BH_FP64], axis=1))))
    finally:
        gpu.set_precision(bl.BH_FP32)
    print("median error", np.exp(np.mean(log)), flush=True)
    assert np.exp(np.mean(log)) <= WHOLE[case]
