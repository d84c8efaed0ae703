"""Walk units taken from other queues than a wavefront's own.

A batch whose first systems hold nearly all of the work (large ones, then many
of one to a few dozen particles) leaves most wavefronts without units early;
fewer units than wavefronts, and hardly more, are the other ends. Every system
keeps the bytes of its step alone, and every particle is stepped once."""
import numpy as np
import pytest

from bhgpu import ic, layout
from bhgpu import lib as bl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [bl.BH_FP32, bl.BH_FP64])
@pytest.mark.parametrize("sizes", [[3], [20000] + [1] * 3000, [24] * 6000, [1] * 700 + [60000] + [17] * 5000,
                                   [70000, 30, 70000, 30, 900]])
def test_uneven_queues(gpu, sizes, prec):
    fp = layout.force_params(0.5, 1e-4, 1.0, True)
    parts = [ic.plummer(n, 11 + n) if n > 1 else ic.random_box(1, 5, 1.0) for n in sizes]
    table = np.concatenate([layout.system(len(q), fp, 8, 64, 16, 1e-3, 1e-3) for q in parts])
    print(f"queues {len(sizes)} systems, prec {prec}", flush=True)
    gpu.set_precision(prec)
    try:
        out, _ = gpu.step_batch(np.concatenate(parts), table)
        lo, seen = 0, {}
        for q in parts:
            if len(q) not in seen:
                seen[len(q)] = gpu.step(q, fp, 8, 64, 16, 1e-3, 1e-3)[0].tobytes()
            assert out[lo:lo + len(q)].tobytes() == seen[len(q)], len(q)
            lo += len(q)
    finally:
        gpu.set_precision(bl.BH_FP32)
