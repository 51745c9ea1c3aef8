"""The host half of scene creation (scene_prep.cpp, bvh_build.cpp; no GPU):
refusals, and inputs that its recursions must end on."""
import ctypes as C
import multiprocessing as mp
import os
import subprocess

import numpy as np
import pytest

from povray_amd import _abi as A
from povray_amd import scenes

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "povray_amd", "csrc")


@pytest.fixture(scope="module")
def prep(tmp_path_factory):
    """prep(scene) -> (status, message, ms, sizes)"""
    so = str(tmp_path_factory.mktemp("prep") / "prep_check.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-ffp-contract=off", "-shared",
                           os.path.join(HERE, "prep_check.cpp")] +
                          [os.path.join(CSRC, f) for f in ("scene_prep.cpp", "bvh_build.cpp", "kd_build.cpp")] +
                          ["-o", so, "-lpthread"])
    L = C.CDLL(so)

    def call(scene):
        desc, keep = scene.desc()
        ms, sizes, msg = C.c_double(), (C.c_uint64 * 4)(), C.create_string_buffer(256)
        rc = L.prep(C.byref(desc), None, C.byref(ms), sizes, msg)
        del keep
        return rc, msg.value.decode(), ms.value, list(sizes)

    return call


def _spheres(nodes, kids, roots, n=2):
    objects = np.array([[A.PVX_CSG, r, 0, 0] for r in roots] + [[A.PVX_SPHERE, 0, 0, 0]], np.uint32)
    return scenes.Scene(name="csg", objects=objects, sphere_center=np.arange(3.0 * n).reshape(-1, 3),
                        sphere_radius=np.ones(n), csg=np.array(nodes, np.uint32),
                        csg_children=np.array(kids, np.uint32),
                        camera=scenes.look_at_camera((0.0, 0.0, -9.0), (0.0, 0.0, 0.0), 16, 12))


def _in_child(fn, want):
    # a child process: a recursion without end fails the test, not the run
    p = mp.get_context("fork").Process(target=lambda: os._exit(0 if fn() == want else 1))
    p.start()
    p.join(20)
    if p.is_alive():
        p.kill()
        p.join()
    assert p.exitcode == 0


SPHERE, CSG = [A.PVX_SPHERE, 0, 0, 0], lambda k: [A.PVX_CSG, k, 0, 0]  # noqa: E731


@pytest.mark.parametrize("op", [A.PVX_CSG_UNION, A.PVX_CSG_INTERSECTION, A.PVX_CSG_MERGE])
def test_cycle_of_csg_nodes(prep, op):
    # nodes 0 and 1 contain each other, node 2 itself; node 3 is a plain one
    nodes = [[op, 0, 2, 0], [op, 2, 2, 0], [op, 4, 2, 0], [op, 6, 1, 0]]
    kids = [CSG(1), SPHERE, CSG(0), SPHERE, CSG(2), SPHERE, SPHERE]
    _in_child(lambda: prep(_spheres(nodes, kids, [3]))[0], 0)  # no object refers to the cycles
    for root in (0, 2):
        _in_child(lambda: prep(_spheres(nodes, kids, [root]))[:2], (1, "a nested CSG node is listed as a top-level object"))


def _holes(n):
    """A box minus n spheres: one CSG object, an intersection of n + 1 operands."""
    r = np.random.default_rng(1)
    kids = [[A.PVX_BOX, 0, 0, 0]] + [[A.PVX_SPHERE, k, A.PVX_FLAG_INVERTED, 0] for k in range(n)]
    return scenes.Scene(
        name="holes", objects=np.array([[A.PVX_CSG, 0, 0, 0]], np.uint32), sphere_center=r.uniform(-4.0, 4.0, (n, 3)),
        sphere_radius=np.full(n, 0.2), box_corner1=np.array([[-4.0, -4.0, -4.0]]),
        box_corner2=np.array([[4.0, 4.0, 4.0]]), box_transform=np.array([-1], np.int32),
        csg=np.array([[A.PVX_CSG_INTERSECTION, 0, n + 1, 0]], np.uint32), csg_children=np.array(kids, np.uint32),
        camera=scenes.look_at_camera((0.0, 0.0, -12.0), (0.0, 0.0, 0.0), 16, 12))


def test_wide_difference_is_linear(prep):
    # eight times the operands: eight times the work and a little more for the
    # deeper tree, not sixty-four times
    ms = []
    for n in (1000, 8000):
        s, best = _holes(n), 1e9
        for _ in range(5):
            rc, msg, t, sizes = prep(s)
            assert rc == 0 and sizes[0] == n + 1, msg
            best = min(best, t)
        ms.append(best)
    assert ms[1] < 24.0 * ms[0]


def test_no_threads_left(prep):
    # a stack size that no thread can have: std::thread throws, the tree is
    # built all the same
    s = scenes.sphere_scene(n=100000)
    want = prep(s)[3]

    def starved():
        attr, L = C.create_string_buffer(64), C.CDLL(None)
        L.pthread_attr_setstacksize.argtypes = [C.c_void_p, C.c_size_t]
        L.pthread_attr_init(attr)
        assert L.pthread_attr_setstacksize(attr, 1 << 46) == 0
        assert L.pthread_setattr_default_np(attr) == 0
        rc, msg, _, sizes = prep(s)
        return rc, sizes

    _in_child(starved, (0, want))
