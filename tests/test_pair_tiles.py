"""How the narrowphase launch shares out its LDS and its test lists: a host build of the rules the kernel uses."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not available")


@pytest.fixture(scope="module")
def violations(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("native") / "pair_tiles_check")
    subprocess.run(["hipcc", "-x", "hip", "--offload-arch=gfx950", "-O2", "-std=c++17", "-Wno-unused-result",
                    "-I", os.path.join(ROOT, "reactphysics3d_amd", "csrc"),
                    os.path.join(HERE, "native", "pair_tiles_check.cpp"), "-o", exe], check=True, capture_output=True)
    out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout
    return {line.split()[0]: int(line.split()[1]) for line in out.splitlines()}


def test_a_wavefront_keeps_to_its_part_of_the_lds(violations):
    assert violations["lds"] == 0


def test_every_pair_of_a_list_is_in_one_share(violations):
    assert violations["shares"] == 0


def test_the_grid_has_a_workgroup_for_every_tile_of_a_shorter_list(violations):
    assert violations["grid"] == 0
