"""The rule for two groups of waves per tile of the weights-direct forward kernel, on the CPU: not on a K so short that they are
slower than one group, which differs by the tile, and never with several workgroups to a unit."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TILES = ("128x128", "128x256", "gate_up")


@pytest.fixture(scope="module")
def groups(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host") / "fwd_k_groups")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "latentq_llm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "fwd_k_groups.cpp"), "-o", exe], check=True)

    def run(tile, workgroups, K, cus=256):
        r = subprocess.run([exe], input="%d %d %d %d" % (TILES.index(tile), workgroups, cus, K), capture_output=True, text=True, check=True)
        return int(r.stdout)
    return run


# the longest K on which two groups measured slower than one by more than the runs differ, and the shortest on which they are faster
@pytest.mark.parametrize("tile,workgroups,slower,faster", [("128x128", 160, 768, 1024), ("128x128", 256, 768, 1024), ("128x256", 128, 1280, 1536),
                                                           ("128x256", 64, 1280, 1536), ("gate_up", 128, 2560, 3072), ("gate_up", 160, 2560, 3072),
                                                           ("gate_up", 240, 2560, 3584), ("gate_up", 256, 3840, 6144)])
def test_two_groups_where_they_are_faster(groups, tile, workgroups, slower, faster):
    assert groups(tile, workgroups, slower) == 1 and groups(tile, workgroups, 256) == 1
    assert groups(tile, workgroups, faster) == 2 and groups(tile, workgroups, 16384) == 2
    assert groups(tile, 257, 16384) == 1 and groups(tile, workgroups, 16384, cus=workgroups - 1) == 1
