"""The position correction of joints runs on two lanes a joint, with the bodies in LDS or not by their number.
Towers of every joint kind with limits, motors and locked axes step to the same bits alone, beside bodies
enough to leave LDS, in a batch of several worlds to a group, and in the per-colour layout."""
import numpy as np
import pytest

from reactphysics3d_amd import scene as S

pytestmark = pytest.mark.gpu

LIMITS = {S.HINGE: (1, (-0.1, 0.1, 0.0, 0.0)), S.SLIDER: (3, (-0.1, 0.1, 0.5, 2.0)),
          S.BALLSOCKET: (1, (0.2, 0.0, 0.0, 0.0)), S.FIXED: (0, (0.0, 0.0, 0.0, 0.0))}


def _scene(towers, baumgarte, spare=0):
    """Towers joined in the air (no contacts), every third tower's kinds in another order."""
    kinds = (S.HINGE, S.FIXED, S.SLIDER, S.BALLSOCKET)
    limits = {k: (f | (4 if baumgarte else 0), v) for k, (f, v) in LIMITS.items()}
    sc = None
    for t in range(towers):
        sc = S.jointed_tower(5 + t % 7, seed=9 + t, kinds=kinds[t % 3:] + kinds[:t % 3], origin=(6.0 * t, 0.0), sc=sc,
                             with_ground=False, limits=limits)
    sc.add_body(S.DYNAMIC, (-9.0, 0.0, 0.0), llock=(1.0, 0.5, 0.0), alock=(0.0, 1.0, 1.0), ang=(1.0, 2.0, 3.0))
    sc.add_joint(S.FIXED, 0, len(sc.bodies) - 1, (-5.0, 0.0, 0.0))
    for i in range(spare):
        sc.add_body(S.DYNAMIC, (3.0 * (i % 50), 3.0 * (i // 50), 500.0))
    return sc


def _run(scenes, n, **kw):
    from reactphysics3d_amd.lib import Batch
    dev = Batch(scenes, **kw)
    dev.step(1.0 / 60.0, 25)
    return [a[:n].copy() for a in dev.bodies()]


# one joint a slot; more joints in a slot than the workgroup's 32 pairs of lanes
@pytest.mark.parametrize("towers", [1, 75])
@pytest.mark.parametrize("baumgarte", [False, True])
def test_every_layout_gives_the_same_bits(towers, baumgarte):
    sc = _scene(towers, baumgarte)
    n = len(sc.bodies)
    want = _run(sc, n, solver="fused", fused_block=64)
    assert all(np.isfinite(a).all() for a in want)
    for got in (_run(_scene(towers, baumgarte, spare=2600), n, solver="fused"),
                _run([sc, _scene(1, baumgarte)], n, solver="fused", group_bodies=4096),
                _run(sc, n, solver="per_color")):
        for a, b in zip(want, got):
            assert np.array_equal(a, b)
