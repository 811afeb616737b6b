"""The broadphase's collider order keeps its tiles small when some bodies are far from the others: a host build of
the rule the kernel uses.  A tile of 64 meets few others, about as many with bodies fallen far out of the scene as
without; with the extents of all bodies' extremes it met all of them."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not available")


@pytest.fixture(scope="module")
def meets(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("native") / "strip_order_check")
    subprocess.run(["hipcc", "-x", "hip", "--offload-arch=gfx950", "-O2", "-std=c++17", "-Wno-unused-result",
                    "-I", os.path.join(ROOT, "reactphysics3d_amd", "csrc"),
                    os.path.join(HERE, "native", "strip_order_check.cpp"), "-o", exe], check=True, capture_output=True)
    return lambda *a: float(subprocess.run([exe, *map(str, a)], capture_output=True, text=True, check=True).stdout.split()[0])


@pytest.mark.parametrize("scene,most", [("heap", 10), ("row", 5), ("mound", 22)])
@pytest.mark.parametrize("far", [0, 1, 20, 1000])   # of 20,000
def test_far_bodies_leave_the_tiles_small(meets, scene, far, most):
    assert 1.0 <= meets(scene, far) <= most


def test_extremes_would_not(meets):
    assert meets("heap", 20, "extremes") > 300   # of 313 tiles
