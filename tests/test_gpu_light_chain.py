"""Light rays followed through glass in the walk, the bounces of a frame
together: frames against the oracle's TraceRay and against light rays followed
a layer a launch (the kd-tree's frames), image and light-ray count, with area
lights (several light rays a hit), supersampling, more layers in a row than
are followed, and light rays followed in the middle of a frame."""
import ctypes as C

import numpy as np
import pytest

from oracle.oracle import OracleScene
from povray_amd import _abi as A
from povray_amd import hip, scenes

pytestmark = pytest.mark.gpu


def _q(a):
    return np.round(np.clip(a, 0.0, 1.0) * 255.0).astype(np.int32)


def _close(img, ref):
    # the parity bar of the shaded frames: 1/255 on 99.9 % of the pixels
    assert np.mean(np.abs(_q(img) - _q(ref)).max(-1) <= 1) >= 0.999


def _layers(n, lights):
    """n glass boxes in a row between the light and a floor, a torus among
    them (the walk of any primitive kind)."""
    c1 = np.array([[-2.0, 0.5 + 0.1 * k, -2.0] for k in range(n)])
    objects = [[A.PVX_BOX, k, 0, 0] for k in range(n)] + [[A.PVX_TORUS, 0, 0, 0], [A.PVX_PLANE, 0, 0, 0]]
    m = len(objects)
    glass = np.arange(m) < n
    return scenes.Scene(
        name=f"layers{n}", objects=np.array(objects, np.uint32), box_corner1=c1, box_corner2=c1 + [[4.0, 0.05, 4.0]],
        box_transform=np.full(n, -1, np.int32), torus_major=np.array([1.0]), torus_minor=np.array([0.2]),
        torus_transform=np.array([0], np.int32), torus_sturm=np.array([1], np.uint8),
        transforms=np.array([scenes._xf_row(scenes.translation_transform([0.0, 0.25, 0.0]))]),
        plane_normal=np.array([[0.0, 1.0, 0.0]]), plane_distance=np.array([0.0]),
        camera=scenes.look_at_camera((0.0, 0.35, -6.0), (0.0, 0.2, 0.0), 96, 54), lights=lights,
        materials=dict(pigment=np.full((m, 3), 0.9), diffuse=np.full(m, 0.6), ambient=np.full(m, 0.05),
                       phong=np.zeros(m), phong_size=np.full(m, 40.0), reflection=np.zeros(m), ior=np.ones(m),
                       transmit=np.where(glass, 0.8, 0.0), filter=np.where(glass, 0.15, 0.0)),
        settings=dict(max_trace_level=6, adc_bailout=1.0 / 255.0))


POINT = [dict(kind="point", position=np.array([0.5, 20.0, -0.3]), colour=np.ones(3))]
AREA = [dict(kind="area", position=np.array([0.0, 12.0, 0.0]), axis1=np.array([2.0, 0.0, 0.0]),
             axis2=np.array([0.0, 0.0, 2.0]), size=(3, 4), colour=np.ones(3))]


# a light ray meets two surfaces a box and is followed through at most 64: 33
# boxes and more end it on the way
@pytest.mark.parametrize("n,lights", [(1, POINT), (20, POINT), (31, POINT), (32, POINT), (33, POINT), (40, POINT),
                                      (70, POINT), (6, AREA), (3, POINT + AREA)])
def test_layers(gpu, n, lights):
    s = _layers(n, lights)
    g, steps = gpu.GpuScene(s), gpu.GpuScene(s, accel=A.PVX_ACCEL_BSP)
    g.set_shading()
    steps.set_shading()
    img, st = g.render()
    ref, _ = OracleScene(s).render(s)
    _close(img, ref)
    by_layer, sst = steps.render()  # light rays followed a layer a launch
    assert np.array_equal(img, by_layer)
    assert st["shadow_rays"] == sst["shadow_rays"] and st["closest_rays"] == sst["closest_rays"]
    if lights is POINT and n >= 33:  # some light rays of the floor were followed to the limit
        assert st["shadow_rays"] > 64 * 96
    again, st2 = g.render()
    assert np.array_equal(img, again) and st2["shadow_rays"] == st["shadow_rays"]


def test_supersampled_glass_field(gpu):
    s = scenes.csg_scene(n_objects=400, width=64, height=36)
    offs = gpu.m1_offsets()
    g = gpu.GpuScene(s)
    g.set_shading()
    img, _ = g.render_samples(offs)
    ref, _ = OracleScene(s).render(s, offsets=offs)
    _close(img, ref)


def _free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    hip.check(hip._lib().hipMemGetInfo(C.byref(free), C.byref(total)), "hipMemGetInfo")
    return free.value


def test_waiting_light_rays_are_bounded(gpu):
    # 64 lights: a hit keeps 1.3 KB and its light rays 4.6 KB.  One frame's
    # worth is 85 MB, and the hits that wait beyond it at most 256 MB.
    lights = [dict(kind="point", position=np.array([0.5 * k, 20.0, -0.3]), colour=np.full(3, 1.0 / 64)) for k in range(64)]
    s = _layers(3, lights)
    g = gpu.GpuScene(s)
    g.set_shading()
    g.render(32, 18)  # the scene's fixed buffers
    free = _free_bytes()
    g.render(160, 90)
    assert free - _free_bytes() < (256 + 85 + 100) << 20


def _many_lights(n, w, h):
    """A glass frame whose hits keep so much (`n` lights) that only a few
    frames' worth wait: light rays are followed in the middle of the frame."""
    s = scenes.csg_scene(n_objects=1000, width=w, height=h)
    r = np.random.default_rng(4)
    s.lights = [dict(kind="point", position=p, colour=np.full(3, 1.0 / n)) for p in r.uniform(-30.0, 30.0, (n, 3))]
    return s


def test_light_rays_followed_mid_frame(gpu):
    # 256 lights: a hit keeps 24 KB, 256 MB hold 2.2 more frames' worth of 96 x
    # 54 rays.  Against light rays followed a layer a launch, which waits for
    # none (the kd-tree's frames): image and light-ray count.  The light rays
    # are followed between a bounce's closest hits and the read-back of their
    # time, which must not take the light rays' for its own (all is on one
    # stream, so the two sums are parts of the frame).
    s = _many_lights(256, 96, 54)
    g, steps = gpu.GpuScene(s), gpu.GpuScene(s, accel=A.PVX_ACCEL_BSP)
    g.set_shading()
    steps.set_shading()
    ref, rst = steps.render()
    for _ in range(2):
        img, st = g.render()
        assert st["closest_rays"] > 3.2 * 96 * 54
        assert np.array_equal(img, ref)
        assert st["shadow_rays"] == rst["shadow_rays"] and st["closest_rays"] == rst["closest_rays"]
        assert st["trace_ms"] + st["shadow_ms"] <= 1.01 * st["total_ms"]
