"""The tile broadphase (index order up to 8,192 colliders, strips beyond) lists the same oriented pairs as
the per-world box scan, step after step: sizes around a tile, several worlds per tile, more colliders
than the index order takes, moving bodies that overlap more colliders than a slab holds, and bodies far from the
others."""
import numpy as np
import pytest

from reactphysics3d_amd import scene as S

pytestmark = pytest.mark.gpu


def _heap(n, seed):
    side = max(6.0, float(np.sqrt(n * 0.6)))
    return S.mixed_container(n, extent=(side, side, 12.0), seed=seed)


def _spread(n, seed):
    """A heap of n bodies, a twentieth of them far away in all directions, two beyond what a float resolves."""
    sc = _heap(n, seed)
    rng = np.random.default_rng(seed)
    for i in range(5, len(sc.bodies), 20):   # (a floor and four walls first)
        b = list(sc.bodies[i])
        b[1] = tuple(float(x) for x in rng.normal(size=3) * 10.0 ** rng.uniform(2.0, 6.0))
        sc.bodies[i] = tuple(b)
    for i, x in ((6, 3e18), (7, -3e18)):
        if i < len(sc.bodies):
            sc.bodies[i] = (sc.bodies[i][0], (x, x, x)) + tuple(sc.bodies[i][2:])
    return sc


def _plate(n, seed):
    """A heap of n bodies with a wide kinematic plate as the first body: it overlaps most of them at once."""
    heap = _heap(n, seed)
    sc = S.Scene(f"plate_{n}", heap.settings)
    p = sc.add_body(S.KINEMATIC, (0.0, 0.0, 6.0), lin=(0.1, 0.0, 0.0))
    sc.add_collider(p, S.BOX, (6.0, 6.0, 5.0))
    sc.bodies += heap.bodies
    sc.colliders += [(c[0] + 1,) + tuple(c[1:]) for c in heap.colliders]
    return sc


def _crowd(n, seed):
    """n bodies that each overlap some 100 others, among them a compound of 80 overlapping parts."""
    rng = np.random.default_rng(seed)
    sc = S.Scene("crowd", S.make_settings(gravity=(0.0, 0.0, 0.0)))
    side = 1.2 * (n / 100.0 * 4.2) ** (1.0 / 3.0)
    parts = sc.add_body(S.DYNAMIC, (side / 2, side / 2, side / 2))
    for p in rng.uniform(-0.3, 0.3, (80, 3)):
        sc.add_collider(parts, S.SPHERE, (0.4,), lpos=tuple(p), trigger=True)
    for p, v in zip(rng.uniform(0.0, side, (n, 3)), rng.normal(size=(n, 3))):
        b = sc.add_body(S.KINEMATIC, tuple(p), lin=tuple(v))
        sc.add_collider(b, S.SPHERE, (0.5,))
    return sc


@pytest.mark.parametrize("name,worlds", [
    ("one", lambda: [_heap(1, 3)]),
    ("tile edge", lambda: [_heap(59, 3), _heap(58, 4), _heap(1, 5)]),
    ("tiles", lambda: [_heap(700, 6)]),
    ("plate over a slab", lambda: [_plate(150, 7), _plate(64, 8)]),
    ("plates, many", lambda: [_plate(400, 9 + k) for k in range(4)]),
    ("strips", lambda: [_heap(380, 20 + k) for k in range(22)] + [_plate(300, 50)]),
    ("crowd", lambda: [_crowd(700, 60)]),
    ("crowds, strips", lambda: [_crowd(600, 61 + k) for k in range(13)]),
    ("strips, far bodies", lambda: [_spread(380, 20 + k) for k in range(23)]),
], ids=lambda x: x if isinstance(x, str) else "")
def test_tiles_list_the_scans_pairs(name, worlds):
    from reactphysics3d_amd.lib import Batch
    scenes = worlds()
    a = Batch(scenes, solver="fused", broadphase="tree", pairs_per_collider=96)
    b = Batch(scenes, solver="fused", broadphase="world_scan", pairs_per_collider=96)
    for k in range(12):
        a.step(1.0 / 60.0)
        b.step(1.0 / 60.0)
        for x, y in zip(a.pairs(), b.pairs()):
            assert np.array_equal(x, y), f"step {k}: pairs differ"
    for x, y in zip(a.bodies(), b.bodies()):
        assert np.array_equal(x, y)


# 64 partners fill a slab, 1,024 the list that is sorted in LDS; beyond 8,192 colliders the order is by strips and that
# list is collected by tiles
@pytest.mark.parametrize("inside,outside", [(63, 200), (64, 200), (65, 200), (1023, 200), (1024, 200), (1025, 200),
                                            (64, 8300), (65, 8300), (300, 8300), (1024, 8300), (1025, 8300), (9000, 200)])
def test_a_body_lists_everything_inside_it(inside, outside):
    from reactphysics3d_amd.lib import Batch
    sc = S.Scene("inside", S.make_settings(gravity=(0.0, 0.0, 0.0)))
    plate = sc.add_body(S.KINEMATIC, (0.0, 0.0, 0.0))
    sc.add_collider(plate, S.BOX, (80.0, 80.0, 1.0))
    for i in np.random.default_rng(inside).permutation(inside + outside):
        b = sc.add_body(S.DYNAMIC, (1.5 * (i % 100) - 75.0, 1.5 * (i // 100) - 70.0, 0.0 if i < inside else 9.0))
        sc.add_collider(b, S.SPHERE, (0.5,), trigger=True)
    dev = Batch(sc, solver="per_color")
    for _ in range(2):
        dev.step(1.0 / 60.0)
        a, b = dev.pairs()
        partners = np.where(a == 0, b, a)[(a == 0) | (b == 0)]
        low = np.array([c for c in range(1, inside + outside + 1) if sc.bodies[c][1][2] == 0.0])
        assert np.array_equal(partners, low)


@pytest.mark.parametrize("kw", [dict(solver="per_color"), dict(solver="fused", broadphase="tree"), dict(solver="fused")])
def test_worlds_without_colliders_step(kw):
    from reactphysics3d_amd.lib import Batch
    sc = S.Scene("points", S.make_settings(gravity=(0.0, 0.0, -10.0)))
    for i in range(5):   # (no collider, no mass: gravity leaves them alone)
        sc.add_body(S.DYNAMIC, (3.0 * i, 0.0, 0.0), lin=(0.0, 0.5, 0.25))
    dev = Batch([sc, sc], **kw)
    dev.step(1.0 / 64.0, 8)
    p = dev.bodies()[0]
    want = np.array([(3.0 * (i % 5), 0.5 * 8 / 64, 0.25 * 8 / 64) for i in range(10)], np.float32)
    assert np.array_equal(p, want) and len(dev.pairs()[0]) == 0   # (exact in FP32)
