"""The ring of scales and zeros of the staged forward kernel, walked on the CPU (lq_staged_ring.h is plain arithmetic): for every
slice of a row that the planner can cut, each piece that a stage reads has arrived and none is requested into its place between
the two barriers in which it is read."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host") / "staged_ring")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "latentq_llm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "staged_ring.cpp"), "-o", exe], check=True)

    def run(slices):
        text = "".join("%d %d %d %d\n" % s for s in slices)
        r = subprocess.run([exe], input=text, capture_output=True, text=True)
        assert r.returncode == 0, r.stdout
        assert r.stdout == "%d slices\n" % len(slices)
    return run


def _slices(groups, per):
    """The slices of a row, in every form the kernel has: pieces of one group, of four (odd rows) or eight, stages of one group or two"""
    for q_log in (0, 2 if groups % 2 else 3):
        for pairs in (0, 1):
            for first in range(0, groups, per):
                yield q_log, pairs, first, min(first + per, groups)


@pytest.mark.parametrize("lo,hi", [(1, 40), (40, 80), (80, 130)])
def test_every_slice_of_every_row(walk, lo, hi):
    # a slice has at least four groups, but for the last one
    walk([s for groups in range(lo, hi) for per in sorted({groups, *range(4, groups)}) for s in _slices(groups, per)])


@pytest.mark.parametrize("N,K", [(2048, 5504), (2048, 5760), (1536, 4224), (1280, 3456), (3328, 9088), (1024, 5504), (4352, 2688)])
def test_slices_the_planner_cuts(walk, hip_lib, N, K):
    """Rows of an odd number of groups with slices that begin at an odd one."""
    from latentq_llm_amd import ops
    groups, odd = K // 128, 0
    for M in range(17, 520):
        kernel, splits, steps = ops.a16w4_plan(M, (N, K), workspace_bytes=64 << 20, compute_units=256)
        if kernel == "staged_128x128":
            per = steps // 2 if splits > 1 else groups
            assert per >= 4 or per == groups
            walk(list(_slices(groups, per)))
            odd += splits > 1 and per % 2
    assert odd
