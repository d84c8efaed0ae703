"""Walk units in pieces, by system size and target size.

A piece walks its unit's or target's box and list for its own particles, so
lists (exact) and forces (1e-12 FP64, 1e-5 FP32 against the FP64 oracle, the
walk's bars) are those of the whole unit, at each class's edges and for
targets that a cut falls into. Above the largest class, where the oracle is
slow, the grouped walk is compared with the per-target walk on the GPU: equal
lists, forces within twice the FP32 bar."""
import numpy as np
import pytest

from bhgpu import ic, layout
from bhgpu import lib as bl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ml,ts", [(300, 4, 16), (4096, 32, 256), (4097, 8, 33), (16384, 16, 32),
                                     (16385, 20, 40), (65536, 40, 100), (65537, 8, 32), (70000, 64, 256)])
def test_units_by_size(gpu, orc, n, ml, ts):
    p = ic.hernquist(n, 31)
    fp = layout.force_params(0.6, 1e-4, 1.0, True)
    oa, opp, opc, otot = orc.build(p, ml, 256).grouped_pass(fp, ts)
    try:
        gpu.build_tree(p, ml, 256)
        for mode in (bl.BH_WALK_GROUPED, bl.BH_WALK_PER_TARGET):
            for prec, tol in ((bl.BH_FP64, 1e-12), (bl.BH_FP32, 1e-5)):
                print(f"units n={n} ml={ml} ts={ts} mode={mode} prec={prec}", flush=True)
                gpu.set_walk_mode(mode)
                gpu.set_precision(prec)
                ga, gpp, gpc, gtot = gpu.accel(fp, ts)
                assert np.array_equal(gpp, opp) and np.array_equal(gpc, opc) and np.array_equal(gtot, otot)
                assert np.sqrt(((ga - oa) ** 2).sum() / (oa ** 2).sum()) < tol
    finally:
        gpu.set_walk_mode(bl.BH_WALK_GROUPED)
        gpu.set_precision(bl.BH_FP32)


def test_largest_units(gpu):
    p = ic.uniform_cube((2 << 20) + 77, 5)
    fp = layout.force_params(0.7, 1e-6, 1.0, True)
    gpu.build_tree(p, 32, 256)
    try:
        ga, gpp, gpc, gtot = gpu.accel(fp, 32)
        gpu.set_walk_mode(bl.BH_WALK_PER_TARGET)
        pa, ppp, ppc, ptot = gpu.accel(fp, 32)
    finally:
        gpu.set_walk_mode(bl.BH_WALK_GROUPED)
    assert np.array_equal(gpp, ppp) and np.array_equal(gpc, ppc) and np.array_equal(gtot, ptot)
    assert np.sqrt(((ga - pa) ** 2).sum() / (pa ** 2).sum()) < 2e-5
