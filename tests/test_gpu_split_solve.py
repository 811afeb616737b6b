"""A large world alone in a fused batch is solved by launches over the whole chip, one beside another world by a
workgroup: the same rows in the same order give the same bits, eagerly and captured, when the colours grow
between capture and replay, and with Baumgarte contacts."""
import numpy as np
import pytest

from reactphysics3d_amd import scene as S

pytestmark = pytest.mark.gpu

DT = 1.0 / 60.0


def _heap(n):
    side = max(6.0, float(np.sqrt(n * 0.6)))
    return S.mixed_container(n, extent=(side, side, 12.0), seed=11)


def _run(scenes, n, steps, graph, baumgarte):
    from reactphysics3d_amd.lib import Batch
    dev = Batch(scenes, solver="fused", group_bodies=1)
    dev.set_contacts_baumgarte(baumgarte)
    dev.step(DT, steps)
    (dev.step_graph if graph else dev.step)(DT, steps)
    it = dev.world_iterations()
    return [a[:n].copy() for a in dev.bodies()] + [np.asarray(x)[:1].copy() for x in it]


@pytest.mark.parametrize("n,steps,graph,baumgarte", [(900, 40, False, False), (1500, 25, True, False), (1500, 40, False, True),
                                                     (3400, 30, False, False), (3400, 12, True, False)])
def test_split_solve_gives_the_same_bits(n, steps, graph, baumgarte):
    sc = _heap(n)
    nb = len(sc.bodies)
    alone = _run([sc], nb, steps, graph, baumgarte)
    beside = _run([sc, _heap(1)], nb, steps, graph, baumgarte)
    assert all(np.isfinite(a).all() for a in alone)
    for a, b in zip(alone, beside):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n,frames", [(1500, 40), (3400, 45)])
def test_a_world_captured_while_it_falls(n, frames):
    """Captured from the first step on, two steps a call: the same bits as eager steps through the change to the split
    solve and the growth of its late colours, and in the end as fast as a capture of the landed world (one workgroup
    alone takes 1.6 times as long at 3,000 bodies)."""
    import time
    from reactphysics3d_amd.lib import Batch
    sc = _heap(n)
    falling, landed = Batch(sc, solver="fused"), Batch(sc, solver="fused")
    for k in range(frames):
        falling.step_graph(DT, 2)
        landed.step(DT, 2)
        if k == 20:
            mid = falling.snapshot()
    for a, b in zip(falling.bodies(), landed.bodies()):
        assert np.array_equal(a, b), "captured and eager steps differ"
    ms = []
    for dev in (falling, landed):
        dev.step_graph(DT, 2)   # landed's capture
        t = []
        for _ in range(7):
            t0 = time.perf_counter()
            dev.step_graph(DT, 4)
            t.append(time.perf_counter() - t0)
        ms.append(min(t))
    assert ms[0] < 1.25 * ms[1] or n < 3000, ms
    falling.restore(mid)
    for _ in range(frames - 21):
        falling.step_graph(DT, 2)
    again = Batch(sc, solver="fused")
    again.step(DT, 2 * frames)
    for a, b in zip(falling.bodies(), again.bodies()):
        assert np.array_equal(a, b), "steps after a restore differ"
