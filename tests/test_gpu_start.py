"""The step's first kernels and its report.

Bounds are reduced over chunks of 1,024 particles (4,096 above 262,144): a
non-finite value at any place of any chunk is found, in one system and in one
of a batch, and leaves the context as it was. The report's phases add up."""
import numpy as np
import pytest

from bhgpu import ic, layout
from bhgpu import lib as bl

pytestmark = pytest.mark.gpu
FP = layout.force_params(0.6, 1e-4, 1.0, True)


@pytest.mark.parametrize("n", [1, 2, 1023, 1024, 1025, 5000, 262144, 262145])
def test_nonfinite_is_found(n):
    p = ic.random_box(n, 3, 1.0)
    print(f"start n={n}", flush=True)
    with bl.Context(0) as gpu:
        good, _ = gpu.step(p, FP, 8, 256, 32, 1e-3, 1e-3)
        for k, i in enumerate(sorted({0, n // 2, n - 1, min(n - 1, 1023), min(n - 1, 1024)})):
            bad = p.copy()
            f, a = [("mass", None), ("pos", 0), ("vel", 2), ("pos", 2), ("vel", 0)][k]
            bad[f][(i,) if a is None else (i, a)] = (np.nan, np.inf, -np.inf)[k % 3]
            with pytest.raises(bl.BHError):
                gpu.step(bad, FP, 8, 256, 32, 1e-3, 1e-3)
            if n <= 5000:
                parts = [p, bad, p[: n // 2]]
                table = np.concatenate([layout.system(len(q), FP, 8, 256, 32, 1e-3, 1e-3) for q in parts])
                with pytest.raises(bl.BHError):
                    gpu.step_batch(np.concatenate(parts), table)
        again, _ = gpu.step(p, FP, 8, 256, 32, 1e-3, 1e-3)
    assert again.tobytes() == good.tobytes()


def test_phases_add_up():
    p = ic.plummer(30000, 2)
    with bl.Context(0) as gpu:
        for _ in range(3):
            gpu.step(p, FP, 16, 256, 32, 1e-3, 1e-3)
            st = gpu.last_step_stats()
            phases = [st.sort_ms, st.tree_ms, st.targets_ms, st.walk_ms]
            assert all(x > 0 for x in phases) and abs(sum(phases) - st.step_ms) < 1e-9
            assert st.step_ms < 1e3
            gpu.build_tree(p, 16, 256)
            gpu.accel(FP, 32)
            st = gpu.last_step_stats()
            assert st.sort_ms == st.tree_ms == 0 and st.walk_ms > 0 and st.targets_ms > 0
