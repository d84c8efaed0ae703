"""How long a context sorts by full keys after a step that needed them.

A far particle leaves more particles to a box of the sort's leading bits than
are ordered there, so the step runs again with full keys. The next 64 steps
use them at once, then the leading bits are tried again (after a trial that
failed, twice as many steps later): a context does not stay slower for good,
and no step's bytes depend on it."""
import pytest

from bhgpu import ic, layout
from bhgpu import lib as bl

pytestmark = pytest.mark.gpu

N = 13000
FP = layout.force_params(0.9, 1e-2, 1.0, False)


@pytest.mark.parametrize("graph", [bl.BH_GRAPH_OFF, bl.BH_GRAPH_ON])
def test_full_keys_end(graph):
    near, far, few = ic.random_box(N, 3, 1.0), ic.random_box(N, 3, 1.0), ic.random_box(500, 3, 1.0)
    far["pos"][-1] = (2.0 ** 12, 0.0, 0.0)
    want = {}
    for name, p in (("near", near), ("far", far), ("few", few)):
        with bl.Context(0) as ctx:
            want[name] = ctx.step(p, FP, 16, 256, 32, 1e-3, 1e-3)[0].tobytes()
    with bl.Context(0) as ctx:
        ctx.set_graph_mode(graph)

        def step(name, p):
            out, _ = ctx.step(p, FP, 16, 256, 32, 1e-3, 1e-3)
            assert out.tobytes() == want[name], name
            return ctx.last_step_stats().reruns

        for k in range(3):  # learn node counts and depths, of full keys too
            step("near", near)
            step("far", far)
        print("full keys: plans learnt", flush=True)
        for _ in range(70):  # the far steps' full keys end
            step("near", near)
        assert step("near", near) == 0
        assert step("far", far) == 1
        assert [step("few", few) for _ in range(70)] == [0] * 70  # these have no such keys and do not count
        assert [step("far", far) for _ in range(2)] == [0, 0]
        assert [step("near", near) for _ in range(62)] == [0] * 62
        print("full keys: 64 steps over", flush=True)
        assert step("far", far) == 1  # a trial, which fails
        assert [step("far", far) for _ in range(128)] == [0] * 128
        assert step("far", far) == 1
        assert [step("near", near) for _ in range(257)] == [0] * 257  # the last by leading bits again
        assert step("far", far) == 1
        assert [step("near", near) for _ in range(64)] == [0] * 64
        assert step("far", far) == 1  # and the span is the first one again
