"""Trees deeper than the walks' stack in LDS (persistent grid with a spill
area) and at most as deep (one launch over all rays): chains of spheres whose
sizes and distances halve, and, split by four bins, fall to 2/9, which gives a
tree as deep as their number."""
import numpy as np
import pytest

from oracle.oracle import OracleScene
from povray_amd import _abi as A
from povray_amd import scenes

pytestmark = pytest.mark.gpu


def _chain(n, box):
    x = 8.0 * 0.5 ** np.arange(n, dtype=np.float64)
    objects = np.zeros((n + (1 if box else 0), 4), np.uint32)
    objects[:n, 0] = A.PVX_SPHERE
    objects[:n, 1] = np.arange(n)
    if box:  # a box: the walk of referenced primitives
        objects[n, 0] = A.PVX_BOX
    return scenes.Scene(
        name=f"chain{n}", objects=objects, sphere_center=np.stack([x, np.zeros(n), np.zeros(n)], 1),
        sphere_radius=0.2 * x + 1e-3, box_corner1=np.array([[-1.0, -3.0, -1.0]]) if box else None,
        box_corner2=np.array([[9.0, -2.0, 1.0]]) if box else None,
        box_transform=np.array([-1], np.int32) if box else None,
        camera=scenes.look_at_camera((3.0, 1.5, -9.0), (3.0, 0.0, 0.0), 83, 61))


@pytest.mark.parametrize("n", [2, 23, 25, 27, 45])
@pytest.mark.parametrize("box", [False, True])
def test_chain_of_spheres(gpu, n, box):
    s = _chain(n, box)
    r = np.random.default_rng(n)
    # rays along the chain's axis meet every box of it
    axis = np.concatenate([np.stack([np.full(3000, 20.0), r.normal(0, 0.02, 3000), r.normal(0, 0.02, 3000)], 1),
                           np.tile([[-1.0, 0.0, 0.0]], (3000, 1))], 1)
    rays = np.concatenate([scenes.camera_rays_np(s.camera), axis])
    md = r.uniform(5.0, 25.0, rays.shape[0])
    g, orc = gpu.GpuScene(s), OracleScene(s)
    for kind, dist in ((A.PVX_RAY_IMAGE, None), (A.PVX_RAY_SHADOW, md)):
        c = orc.find_intersection(rays, dist, kind, method=0)
        got = [g.find_intersection(rays, dist, kind),
               gpu.GpuBatch([g]).find_intersection([rays], kind, None if dist is None else [dist])[0]]
        if not box:
            g.set_traversal(A.PVX_TRAVERSAL_BINARY, 1, kind)
            got.append(g.find_intersection(rays, dist, kind))
            g.set_traversal(ray_kind=kind)
        for h in got:
            assert np.array_equal(h["obj"], c["obj"]) and np.array_equal(h["t"], c["t"])
    few = g.find_intersection(rays[-7:])
    assert np.array_equal(few["obj"], orc.find_intersection(rays[-7:], None, A.PVX_RAY_IMAGE, method=0)["obj"])


def _deep(n, box):
    # a split by four bins takes one sphere off: each is below a quarter of the
    # distance of the one before
    s = _chain(n, box)
    x = 8.0 * 4.5 ** -np.arange(n, dtype=np.float64)
    s.sphere_center = np.stack([x, np.zeros(n), np.zeros(n)], 1)
    s.sphere_radius = 0.2 * x
    return s


# depth 24 fits the LDS stack, the others do not
@pytest.mark.parametrize("n,depth", [(25, 24), (26, 25), (27, 26), (40, 39)])
@pytest.mark.parametrize("box", [False, True])
def test_walks_beyond_the_lds_stack(gpu, n, depth, box):
    s = _deep(n, box)
    r = np.random.default_rng(n)
    k = 3000
    far = np.concatenate([np.full((k, 1), 20.0), r.normal(0, 0.02, (k, 2))], 1)
    axis = np.concatenate([np.concatenate([far, np.tile([[-1.0, 0.0, 0.0]], (k, 1))], 1),
                           np.concatenate([far * [-1, 1e-3, 1e-3], np.tile([[1.0, 0.0, 0.0]], (k, 1))], 1)])
    rays = np.concatenate([scenes.camera_rays_np(s.camera), axis])
    md = r.uniform(5.0, 25.0, rays.shape[0])
    g, orc = gpu.GpuScene(s, sah_bins=4), OracleScene(s)
    assert g.stats()["bvh_depth"] == depth
    for kind, dist in ((A.PVX_RAY_IMAGE, None), (A.PVX_RAY_SHADOW, md)):
        c = orc.find_intersection(rays, dist, kind, method=0)
        got = [g.find_intersection(rays, dist, kind), g.find_intersection(rays[-7:], None if dist is None else dist[-7:], kind),
               gpu.GpuBatch([g]).find_intersection([rays], kind, None if dist is None else [dist])[0]]
        if not box:
            for v in (A.PVX_TRAVERSAL_BINARY, A.PVX_TRAVERSAL_BINARY_WW):
                g.set_traversal(v, 1, kind)
                got.append(g.find_intersection(rays, dist, kind))
            g.set_traversal(ray_kind=kind)
        for h in got:
            ref = c[-len(h):]
            assert np.array_equal(h["obj"], ref["obj"]) and np.array_equal(h["t"], ref["t"])


@pytest.mark.parametrize("make,grows", [(lambda: scenes.mesh_scene(level=5, width=64, height=48), False),
                                        (lambda: scenes.radiosity_scene(n_boxes=300, width=64, height=48), False),
                                        (lambda: scenes.csg_scene(n_objects=400, width=64, height=48), False),
                                        (lambda: _deep(40, False), True), (lambda: _deep(40, True), True)])
def test_spill_area_only_for_deep_trees(gpu, make, grows):
    s = make()
    g = gpu.GpuScene(s, sah_bins=4 if grows else 0)
    before = g.stats()["device_bytes"]
    rays = scenes.camera_rays_np(s.camera)
    g.find_intersection(rays)
    g.find_intersection(rays, np.full(rays.shape[0], 9.0), A.PVX_RAY_SHADOW)
    if s.lights:
        g.set_shading()
        g.render()
    assert (g.stats()["device_bytes"] > before + (1 << 20)) == grows
