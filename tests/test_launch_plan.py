"""Launch shapes and scratch sizes worked out on the host (eos_amd/csrc/launch_plan.h),
at sizes up to the largest an entry point takes."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
INT_MAX = 2**31 - 1
STATIC_MAX_RAYS = 1 << 20

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    so = tmp_path_factory.mktemp("plan") / "libplan.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "eos_amd", "csrc"),
                    os.path.join(ROOT, "tests", "plan", "launch_plan.cpp"), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.plan_max_launch_items.restype = C.c_longlong
    return lib


def _linear(plan, n, n_tri, static):
    out = (C.c_longlong * 9)()
    plan.plan_linear(n, n_tri, int(static), out)
    return dict(zip(("lanes", "chunk", "chunks", "runs", "scan_blocks", "merge_blocks", "scan_items", "merge_items",
                     "bytes"), out))


@pytest.mark.parametrize("n", [1, 2, 3, 64, 127, 128, 129, 256, 257, 4000, 20000, 300_000, 2**19 - 1, 2**19, 2**19 + 1,
                               2**20, 2**20 + 1, 2**26 - 1, 2**26, 2**26 + 1, 2**30, INT_MAX])
@pytest.mark.parametrize("static", [False, True])
def test_linear_split(plan, n, static):
    if static and n > STATIC_MAX_RAYS:
        pytest.skip("refused by eos_trace_rays_static")
    limit = plan.plan_max_launch_items()
    for n_tri in (0, 1, 255, 256, 257, 5000, 13312, 1_000_000, 2**28 - 1):
        r = _linear(plan, n, n_tri, static)
        # every ray and every triangle is covered, by launches of a permitted size
        assert r["scan_items"] >= n * r["lanes"] and r["scan_items"] < limit, (n, n_tri, r)
        assert r["chunk"] % 256 == 0 and r["chunk"] * r["chunks"] >= n_tri and 1 <= r["chunks"] <= 65535
        assert r["chunk"] * (r["chunks"] - 1) < max(n_tri, 1)              # no chunk is empty
        assert r["merge_items"] < limit, (n, n_tri, r)
        # one run per ray is kept only where several lanes or chunks share a ray
        if r["chunks"] == 1 and r["lanes"] == 1:
            assert r["runs"] == 0 and r["merge_blocks"] == 0
        else:
            assert r["runs"] == n * r["chunks"] and r["merge_items"] >= 64 * n
            assert r["bytes"] <= (16 if static else 32) * STATIC_MAX_RAYS


@pytest.mark.parametrize("resident", [1, 64, 1280, 4096])
def test_query_stacks(plan, resident):
    out = (C.c_longlong * 2)()
    for n in (1, 2, 63, 64, 65, 100, 255, 256, 257, 1000, 5000, 20000, 81919, 81920, 81921, 1_000_003, INT_MAX):
        plan.plan_query(C.c_longlong(n), resident, out)
        grid, lanes = out
        assert 1 <= grid <= resident and grid * 256 < plan.plan_max_launch_items()
        # a wave beyond the ceil(n / 64) that a ray per lane fills leaves at once; every wave
        # before has room for each of its lanes
        walking = min(4 * grid, (n + 63) // 64)
        assert 64 * walking == lanes, (n, grid, lanes)
        # no more than the rays, but for the last wave
        assert lanes < n + 64


def test_a_callers_knobs_are_taken_as_they_are(plan):
    from eos_amd import _lib as E
    refill, scatter = E.Scene.DEFAULT_LAUNCH["refill"], E.Scene.DEFAULT_LAUNCH["scatter"]
    out = (C.c_int * 4)()
    for r in range(1, 65):
        for s in range(0, 65):
            plan.plan_knobs(r, s, out)
            assert out[0] == s
            assert out[1] == (2 if s == scatter else s)
            assert out[2] == (1 if s == scatter else s)
            assert out[3] == (32 if r == refill else r)
