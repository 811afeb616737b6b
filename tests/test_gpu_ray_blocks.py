"""Raycasts walk a world's colliders in blocks, from LDS when a workgroup's rays share a world: rays of several
worlds interleaved in one call answer like each world's rays alone, over block edges (one collider, 64, 65,
more than a staged chunk), for closest and every hits, with clipped fractions and category masks."""
import numpy as np
import pytest

from reactphysics3d_amd import scene as S

pytestmark = pytest.mark.gpu


def _world(n, seed):
    side = max(6.0, float(np.sqrt(n * 0.6)))
    return S.mixed_container(n, extent=(side, side, 8.0), seed=seed)


@pytest.mark.parametrize("sizes", [(1, 59, 60), (507, 508, 1100)])
def test_interleaved_worlds_answer_like_each_alone(sizes):
    from reactphysics3d_amd.lib import Batch
    dev = Batch([_world(n, 40 + n) for n in sizes])
    rng = np.random.default_rng(5)
    n = 1500
    p1 = rng.uniform(-8, 8, (n, 3)).astype(np.float32)
    p2 = rng.uniform(-8, 8, (n, 3)).astype(np.float32)
    mf = rng.uniform(0.1, 1.2, n).astype(np.float32)
    w = rng.integers(0, len(sizes), n).astype(np.int32)
    mixed = dev.raycast(p1, p2, w, mf)
    every = dev.raycast_all(p1, p2, w, mf)
    assert (mixed[0] >= 0).any() and not dev.raycast(p1, p2, w, mf, mask=0x8000)[3].any()
    for k in range(len(sizes)):
        i = np.nonzero(w == k)[0]
        alone = dev.raycast(p1[i], p2[i], w[i], mf[i])
        for a, b in zip(mixed, alone):
            assert np.array_equal(a[i], b)
        ray, *hits = dev.raycast_all(p1[i], p2[i], w[i], mf[i])
        sel = np.isin(every[0], i)
        assert np.array_equal(i[ray], every[0][sel])
        for a, b in zip(every[1:], hits):
            assert np.array_equal(a[sel], b)
    # the closest hit is among the every-hit list, at its smallest fraction
    for r in np.nonzero(mixed[0] >= 0)[0][:200]:
        f = every[4][every[0] == r]
        assert mixed[3][r] == f.min()
