"""CSG objects in the tree leaf by leaf, and their filter programs, against
whole objects (the kd-tree keeps them whole) and the FP64 oracle; launches of
few rays (fewer rays per wavefront) against one large launch."""
import numpy as np
import pytest

from oracle.oracle import OracleScene
from povray_amd import _abi as A
from povray_amd import scenes

pytestmark = pytest.mark.gpu


def _tree_scene(seed, n_trees, arity, depth, inverted, other):
    """Random CSG trees: 1..arity operands a node, up to `depth` levels, all
    operators, leaves inverted where `inverted` says so; leaves spheres, boxes and tori (either
    solver), placed or not, and half-spaces below discs where `other` says so
    (such trees stay whole)."""
    r = np.random.default_rng(seed)
    sph, rad, b1, b2, btr, tR, tr, ttr, tst = [], [], [], [], [], [], [], [], []
    dc, dn, dr, xf, nodes, kids = [], [], [], [], [], []

    def place(pos):
        t = scenes.compose(scenes.rotation_transform(r.uniform(0, 360, 3)), scenes.translation_transform(pos))
        xf.append(scenes._xf_row(t))
        return len(xf) - 1

    def leaf(pos):
        k = int(r.integers(0, 4 if other else 3))
        p = pos + r.uniform(-0.5, 0.5, 3)
        inv = A.PVX_FLAG_INVERTED if inverted and r.uniform() < 0.25 else 0
        if k == 0:
            sph.append(p)
            rad.append(r.uniform(0.3, 0.8))
            return [A.PVX_SPHERE, len(sph) - 1, inv, 0]
        if k == 1:
            e = r.uniform(0.2, 0.7, 3)
            placed = r.uniform() < 0.6
            b1.append(-e if placed else p - e)
            b2.append(e if placed else p + e)
            btr.append(place(p) if placed else -1)
            return [A.PVX_BOX, len(b1) - 1, inv, 0]
        if k == 2:
            tR.append(r.uniform(0.4, 0.8))
            tr.append(tR[-1] * r.uniform(0.15, 0.5))
            ttr.append(place(p))
            tst.append(int(r.integers(0, 2)))
            return [A.PVX_TORUS, len(tR) - 1, inv, 0]
        dc.append(p)
        dn.append(r.uniform(-1, 1, 3))
        dr.append((1.0, 0.0))
        return [A.PVX_DISC, len(dc) - 1, A.PVX_FLAG_INVERTED, 0]

    def node(level, pos):
        me = len(nodes)
        nodes.append(None)
        n = int(r.integers(1, arity + 1))
        first = len(kids)
        kids.extend([None] * n)
        for k in range(n):
            deeper = level < depth and r.uniform() < 0.55
            kids[first + k] = [A.PVX_CSG, node(level + 1, pos), 0, 0] if deeper else leaf(pos)
        nodes[me] = [int(r.choice([A.PVX_CSG_UNION, A.PVX_CSG_INTERSECTION, A.PVX_CSG_MERGE])), first, n, 0]
        return me

    # a plain sphere holds every root, so that no tree is unbounded
    roots = []
    for _ in range(n_trees):
        pos = r.uniform(-4, 4, 3)
        me = len(nodes)
        nodes.append(None)
        first = len(kids)
        kids.extend([None, None])
        sph.append(pos)
        rad.append(1.5)
        kids[first] = [A.PVX_SPHERE, len(sph) - 1, 0, 0]
        kids[first + 1] = [A.PVX_CSG, node(1, pos), 0, 0]
        nodes[me] = [A.PVX_CSG_INTERSECTION, first, 2, 0]
        roots.append(me)
    objects = np.zeros((n_trees, 4), np.uint32)
    objects[:, 0] = A.PVX_CSG
    objects[:, 1] = roots
    return scenes.Scene(
        name="csg_trees", objects=objects, sphere_center=np.array(sph), sphere_radius=np.array(rad),
        box_corner1=np.array(b1).reshape(-1, 3), box_corner2=np.array(b2).reshape(-1, 3),
        box_transform=np.array(btr, np.int32), torus_major=np.array(tR), torus_minor=np.array(tr),
        torus_transform=np.array(ttr, np.int32), torus_sturm=np.array(tst, np.uint8),
        disc_center=np.array(dc).reshape(-1, 3), disc_normal=np.array(dn).reshape(-1, 3),
        disc_radius=np.array(dr).reshape(-1, 2), disc_transform=np.full(len(dc), -1, np.int32),
        transforms=np.array(xf).reshape(-1, 32), csg=np.array(nodes, np.uint32).reshape(-1, 4),
        csg_children=np.array(kids, np.uint32).reshape(-1, 4),
        camera=scenes.look_at_camera((0.0, 1.0, -13.0), (0.0, 0.0, 0.0), 97, 71))


def _same(a, b):
    for k in ("obj", "prim", "t"):
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("seed,n_trees,arity,depth,inverted,other",
                         [(1, 40, 3, 3, False, False), (2, 30, 4, 6, False, False), (3, 25, 2, 7, True, True),
                          (4, 30, 3, 5, True, False), (5, 1, 1, 1, False, False)])
def test_leaf_by_leaf_equals_whole(gpu, seed, n_trees, arity, depth, inverted, other):
    s = _tree_scene(seed, n_trees, arity, depth, inverted, other)
    rays = scenes.camera_rays_np(s.camera)
    md = np.random.default_rng(seed).uniform(5.0, 20.0, rays.shape[0])
    tree, whole = gpu.GpuScene(s), gpu.GpuScene(s, accel=A.PVX_ACCEL_BSP)
    orc = OracleScene(s)
    for kind, dist in ((A.PVX_RAY_IMAGE, None), (A.PVX_RAY_SHADOW, md)):
        g = tree.find_intersection(rays, dist, kind)
        _same(g, whole.find_intersection(rays, dist, kind))
        _same(g, gpu.GpuBatch([tree]).find_intersection([rays], kind, None if dist is None else [dist])[0])
        if not inverted:  # the reference bounds a union's inverted operand by its box and culls hits outside
            c = orc.find_intersection(rays, dist, kind, method=0)
            bad = (g["obj"] != c["obj"]) | (g["prim"] != c["prim"])
            assert not bad.any()
            hit = c["obj"] >= 0
            assert not hit.any() or (np.abs(g["t"][hit] - c["t"][hit]) / c["t"][hit]).max() <= 1e-5


@pytest.mark.parametrize("make", [lambda: scenes.csg_scene(n_objects=400, width=128, height=128),
                                  lambda: scenes.radiosity_scene(n_boxes=300, width=128, height=128),
                                  lambda: scenes.cone_scene(n=60, width=128, height=128)])
def test_few_rays_equal_many(gpu, make):
    s = make()
    g = gpu.GpuScene(s)
    rays = scenes.camera_rays_np(s.camera)
    rays = np.concatenate([rays] * 40)  # enough to fill the grid
    full = g.find_intersection(rays)
    for n in (1, 2, 63, 64, 65, 1023, 4097, 32769, 131073):
        _same(g.find_intersection(rays[:n]), full[:n])


def test_child_ranges_that_overlap(gpu):
    # nodes whose child ranges share leaves: Inside goes by each node's own operands
    r = np.random.default_rng(9)
    n = 14
    centre, kids = r.uniform(-1.0, 1.0, (n, 3)), []
    for k in range(n):
        kids.append([A.PVX_SPHERE if k % 3 else A.PVX_BOX, k, A.PVX_FLAG_INVERTED if k % 5 == 4 else 0, 0])
    ops = [A.PVX_CSG_UNION, A.PVX_CSG_INTERSECTION, A.PVX_CSG_MERGE]
    nodes = [[ops[i % 3], int(a), int(c), 0]
             for i, (a, c) in enumerate(zip(r.integers(0, n - 4, 12), r.integers(2, 5, 12)))]
    for i, op in enumerate(ops):  # two nodes below each
        kids += [[A.PVX_CSG, 2 * i, 0, 0], [A.PVX_CSG, 2 * i + 1, 0, 0]]
        nodes.append([op, len(kids) - 2, 2, 0])
    roots = [i for i in range(len(nodes)) if i >= 6]
    s = scenes.Scene(
        name="overlap", objects=np.array([[A.PVX_CSG, i, 0, 0] for i in roots], np.uint32),
        sphere_center=centre, sphere_radius=r.uniform(0.5, 1.2, n), box_corner1=centre - 0.6,
        box_corner2=centre + 0.6, box_transform=np.full(n, -1, np.int32), csg=np.array(nodes, np.uint32),
        csg_children=np.array(kids, np.uint32), camera=scenes.look_at_camera((0.0, 0.5, -6.0), (0.0, 0.0, 0.0), 97, 71))
    g, orc = gpu.GpuScene(s), OracleScene(s)
    pts = r.uniform(-2.0, 2.0, (20000, 3))
    for ob in range(len(roots)):
        which = np.full(pts.shape[0], ob, np.uint32)
        assert np.array_equal(g.inside(pts, which), orc.inside(pts, which)), nodes[roots[ob]]


def _no_csg(s):
    s.objects = s.objects[s.objects[:, 0] != A.PVX_CSG]
    return s


# what a scene holds picks its walk: cones, discs, polygons and quadrics alone,
# with CSG, with tori
BY_CONTENT = [("simple", lambda: _no_csg(scenes.cone_scene(n=60, width=97, height=71))),
              ("quadrics", lambda: _no_csg(scenes.cone_scene(n=1, n_discs=3, n_quadrics=40, n_polygons=0, width=97, height=71))),
              ("csg", lambda: scenes.cone_scene(n=60, width=97, height=71)),
              ("torus", lambda: scenes.torus_scene(n=20, width=97, height=71)),
              ("placed", lambda: scenes.placed_mesh_scene(level=2, width=97, height=71))]


@pytest.mark.parametrize("name,make", BY_CONTENT)
def test_walks_by_content(gpu, name, make):
    s = make()
    rays = scenes.camera_rays_np(s.camera)
    r = np.random.default_rng(3)
    md = r.uniform(4.0, 20.0, rays.shape[0])
    g, kd, orc = gpu.GpuScene(s), gpu.GpuScene(s, accel=A.PVX_ACCEL_BSP), OracleScene(s)
    boxes = scenes.radiosity_scene(n_boxes=50, width=64, height=48)  # a batch takes the walk of both
    both = gpu.GpuBatch([g, gpu.GpuScene(boxes)])
    box_rays = scenes.camera_rays_np(boxes.camera)
    for kind, dist in ((A.PVX_RAY_IMAGE, None), (A.PVX_RAY_REFLECTION, None), (A.PVX_RAY_SHADOW, md)):
        h = g.find_intersection(rays, dist, kind)
        _same(h, kd.find_intersection(rays, dist, kind))
        c = orc.find_intersection(rays, dist, kind, method=0)
        assert np.array_equal(h["obj"], c["obj"]) and np.array_equal(h["prim"], c["prim"])
        hit = c["obj"] >= 0
        assert np.abs(h["t"][hit] / c["t"][hit] - 1.0).max(initial=0.0) <= 1e-5
        mds = None if dist is None else [dist, np.full(box_rays.shape[0], 5.0)]
        _same(h, both.find_intersection([rays, box_rays], kind, mds)[0])
        for n in (1, 63, 1025):  # few rays per wavefront
            _same(h[:n], g.find_intersection(rays[:n], None if dist is None else dist[:n], kind))


def test_batch_of_every_walk(gpu):
    made = [make() for _, make in BY_CONTENT]
    rays = [scenes.camera_rays_np(s.camera) for s in made]
    gs = [gpu.GpuScene(s) for s in made]
    for upto in range(1, len(gs) + 1):
        for g, r, h in zip(gs[:upto], rays, gpu.GpuBatch(gs[:upto]).find_intersection(rays[:upto])):
            _same(g.find_intersection(r), h)
