"""Bodies, forces and rays pass between the caller's packed arrays and the device in one kernel or copy, in
parts of a fixed size; a snapshot's arrays are copied in one launch."""
import numpy as np
import pytest

from reactphysics3d_amd import scene as S

pytestmark = pytest.mark.gpu

DT = 1.0 / 60.0


def _free_bodies(n, sleeping=0):
    sc = S.Scene("free", S.make_settings(gravity=(0.0, 0.0, 0.0), sleeping=sleeping))
    for i in range(n):
        b = sc.add_body(S.STATIC if i % 7 == 3 else S.DYNAMIC, (4.0 * (i % 40), 4.0 * (i // 40), 0.0))
        sc.add_collider(b, S.SPHERE, (0.5,))
    return sc


@pytest.mark.parametrize("n", [1, 63, 257, 1000])
def test_bodies_and_forces(n):
    from reactphysics3d_amd.lib import Batch
    dev = Batch([_free_bodies(n), _free_bodies(3)])
    rng = np.random.default_rng(n)
    dynamic = np.array([i % 7 != 3 for i in range(n)] + [True] * 3)
    lin, ang = (rng.normal(size=(n + 3, 3)).astype(np.float32) * dynamic[:, None] for _ in range(2))
    dev.set_bodies(lin=lin, ang=ang)
    p, q, v, w = dev.bodies()
    grid = np.array([(4.0 * (i % 40), 4.0 * (i // 40), 0.0) for i in list(range(n)) + [0, 1, 2]], np.float32)
    assert np.array_equal(p, grid) and np.array_equal(q, np.tile(np.float32([0, 0, 0, 1]), (n + 3, 1)))
    assert np.array_equal(v, lin) and np.array_equal(w, ang)
    f, t = (rng.normal(size=(n + 3, 3)).astype(np.float32) for _ in range(2))
    f[::2] = 0.0
    dev.apply_forces(f)
    dev.apply_forces(f, t)   # adds up
    dev.step(DT)
    mass = 4.0 / 3.0 * np.pi * 0.125   # density 1
    want_v = lin + 2.0 * DT / mass * f * dynamic[:, None]
    want_w = ang + DT / (0.4 * mass * 0.25) * t * dynamic[:, None]
    _, _, v, w = dev.bodies()
    # a few FP32 roundings of values of size |w| <= |ang| + dt |t| / inertia < 3
    assert np.abs(v - want_v).max() < 4e-6 and np.abs(w - want_w).max() < 4e-6


def test_a_force_wakes_a_sleeping_body():
    from reactphysics3d_amd.lib import Batch
    dev = Batch(_free_bodies(70, sleeping=1))
    dev.step(DT, 120)
    dynamic = np.array([i % 7 != 3 for i in range(70)])
    assert np.array_equal(dev.sleeping() != 0, dynamic)
    f = np.zeros((70, 3), np.float32)
    f[64] = (1.0, 0.0, 0.0)
    dev.apply_forces(np.zeros_like(f))
    assert np.array_equal(dev.sleeping() != 0, dynamic)
    dev.apply_forces(f)
    dev.step(DT)
    awake = dynamic & (dev.sleeping() == 0)
    assert np.nonzero(awake)[0].tolist() == [64] and dev.bodies()[2][64, 0] > 0.0


def test_rays_over_more_than_one_part():
    from reactphysics3d_amd.lib import Batch
    dev = Batch(S.mixed_container(40, extent=(8.0, 8.0, 8.0), seed=3))
    rng = np.random.default_rng(1)
    n = (16 << 20) // 64 + 77   # 64 bytes a ray, 16 MiB a part
    p1, p2 = (rng.uniform(-5, 5, (n, 3)).astype(np.float32) for _ in range(2))
    mf = rng.uniform(0.2, 1.0, n).astype(np.float32)
    whole = dev.raycast(p1, p2, np.zeros(n, np.int32), mf)
    parts = [dev.raycast(p1[i:i + 100000], p2[i:i + 100000], None, mf[i:i + 100000]) for i in range(0, n, 100000)]
    assert (whole[0] >= 0).any()
    for k in range(4):
        assert np.array_equal(whole[k], np.concatenate([p[k] for p in parts]))
    with pytest.raises(RuntimeError):
        dev.raycast(p1, p2, np.full(n, 1, np.int32))


def test_the_first_read_back_is_no_slower_than_its_copies():
    """The memory it passes through is there before the first call: 1.5 to 1.7 times a later call, 8 times while its
    pages came with that call."""
    import time
    from reactphysics3d_amd.lib import Batch
    sc = S.Scene("points", S.make_settings(gravity=(0.0, 0.0, 0.0)))
    for i in range(3000):
        sc.add_body(S.DYNAMIC, (float(i % 50), float(i // 50), 0.0))
    warm, dev = Batch([sc] * 20), Batch([sc] * 20)
    for b in (warm, warm, warm):   # (the caller's arrays come from memory that it has used before)
        b.bodies()
    dev.step(DT)
    t = []
    for _ in range(5):
        t0 = time.perf_counter()
        dev.bodies()
        t.append(time.perf_counter() - t0)
    assert t[0] < 4.0 * min(t[1:]), t
