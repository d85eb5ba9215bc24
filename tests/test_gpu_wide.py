"""A queue with few rays for the grid's waves is traversed by whole waves
(sixteen nodes and thirty-two leaves at a time), a longer one by lanes.  The
same frame with 64 traversal blocks per CU (every queue by waves) and with
one (the first bounces' queues by lanes) equals the oracle's bit for bit, on
scenes that fill the wave traversal's lists: rays through the boxes of more
instances than it has slots or list entries for, every primitive kind,
groups of one leaf, near-ties, and more transparent hits than are recorded."""
import numpy as np
import pytest

from ospray_amd import api as A
from ospray_amd import capi as K
from ospray_amd import scenes
from oracle import orc
from test_gpu_bvh import _mixed_scene

pytestmark = pytest.mark.gpu

CH = K.OSP_FB_COLOR | K.OSP_FB_ACCUM | K.OSP_FB_DEPTH | K.OSP_FB_ID_PRIMITIVE | K.OSP_FB_ID_OBJECT | K.OSP_FB_ID_INSTANCE


def _crowd(material):
    """300 overlapping instances of a sphere in a row along the view."""
    rng = np.random.default_rng(9)
    unit, faces = scenes.icosphere(1)
    geoms = [scenes.Geometry("triangles", vertex=unit.astype(np.float32), index=faces.astype(np.uint32),
                             normal=unit.astype(np.float32))]
    insts = [scenes.Instance(0, xfm=(s, 0, 0, 0, s, 0, 0, 0, s, x, y, z)) for s, x, y, z in zip(
        rng.uniform(0.2, 1.0, 300), rng.uniform(-2, 2, 300), rng.uniform(-2, 2, 300), rng.uniform(0, 12, 300))]
    return scenes.Scene("crowd", 64, 48, geoms, [scenes.Model(0, 0)], [[0]], insts, [material],
                        [{"type": "ambient", "intensity": 0.5},
                         {"type": "quad", "position": (-2.0, 6.0, -2.0), "edge1": (4.0, 0.0, 0.0),
                          "edge2": (0.0, 0.0, 4.0), "intensity": 5.0}],
                        {"position": (0.0, 0.0, -6.0), "direction": (0.0, 0.0, 1.0), "up": (0.0, 1.0, 0.0),
                         "fovy": 50.0, "aspect": 64 / 48}, {"pixelSamples": 2, "maxPathLength": 5})


def _sized(sc, w=64, h=48, spp=2):
    sc.width, sc.height = w, h
    sc.renderer = dict(sc.renderer, pixelSamples=spp)
    return sc


SCENES = {
    "crowd": lambda: _crowd({"type": "obj", "kd": (0.6, 0.5, 0.4)}),
    "crowd_glass": lambda: _crowd({"type": "glass", "eta": 1.3}),
    "crowd_thin": lambda: _crowd({"type": "obj", "kd": (0.6, 0.5, 0.4), "d": 0.3}),
    "mixed": lambda: _sized(_mixed_scene()),
    "ties": lambda: _sized(scenes.near_tie_layers(instanced=True)),
}


@pytest.mark.parametrize("bpc", [64, 1])
@pytest.mark.parametrize("name", sorted(SCENES))
def test_frames_equal_the_oracle(hip_device, name, bpc):
    sc = SCENES[name]()
    L = K.lib()
    dev = L.ospGetCurrentDevice()
    A.set_device_param(dev, "traceBlocksPerCU", bpc)
    L.ospDeviceCommit(dev)
    try:
        s = scenes.to_ospray(sc)
        fb = A.framebuffer(sc.width, sc.height, K.OSP_FB_RGBA32F, CH)
        A.render(fb, s.renderer, s.camera, s.world)
        got = [A.map_color(fb, sc.width, sc.height, K.OSP_FB_RGBA32F)] + [
            A.map_channel(fb, c, sc.width, sc.height)
            for c in (K.OSP_FB_DEPTH, K.OSP_FB_ID_PRIMITIVE, K.OSP_FB_ID_OBJECT, K.OSP_FB_ID_INSTANCE)]
    finally:
        A.set_device_param(dev, "traceBlocksPerCU", 12)
        L.ospDeviceCommit(dev)
    ofb, _, _ = orc.render_scene(sc, frames=1, fmt=K.OSP_FB_RGBA32F, channels=CH)
    for a, ch in zip(got, (K.OSP_FB_COLOR, K.OSP_FB_DEPTH, K.OSP_FB_ID_PRIMITIVE, K.OSP_FB_ID_OBJECT,
                           K.OSP_FB_ID_INSTANCE)):
        assert np.array_equal(a, ofb.channel(ch), equal_nan=True), ch
