"""Passes of 2^17 paths or more run the shadow stages on a second stream,
shorter ones on one: around the line, with surfaces and with a volume, the
frame equals the one that overlapShadow false makes, bit for bit.  The second
stream's scratch rows follow the traversal grid."""
import numpy as np
import pytest

from ospray_amd import api as A
from ospray_amd import capi as K
from ospray_amd import scenes
from oracle import orc

pytestmark = pytest.mark.gpu

SCENES = {"surfaces": lambda w, h: scenes.c0(w, h),
          "volume": lambda w, h: scenes.c4(w, h, grid=24, base_period=8)}


@pytest.mark.parametrize("w,h", [(512, 248), (512, 256), (520, 264)])
@pytest.mark.parametrize("name", sorted(SCENES))
def test_both_schedules_make_the_same_frame(hip_device, name, w, h):
    sc = SCENES[name](w, h)
    L = K.lib()
    dev = L.ospGetCurrentDevice()
    frames = []
    try:
        for on in (True, False):
            A.set_device_param(dev, "overlapShadow", on)
            L.ospDeviceCommit(dev)
            s = scenes.to_ospray(sc, {"pixelSamples": 1, "maxPathLength": 6})
            fb = A.framebuffer(w, h, K.OSP_FB_RGBA32F, K.OSP_FB_COLOR | K.OSP_FB_ACCUM)
            for _ in range(2):
                A.render(fb, s.renderer, s.camera, s.world)
            frames.append(A.map_color(fb, w, h, K.OSP_FB_RGBA32F))
    finally:
        A.set_device_param(dev, "overlapShadow", True)
        L.ospDeviceCommit(dev)
    assert np.array_equal(frames[0], frames[1])


@pytest.mark.parametrize("first,then", [(1, 12), (4, 16)])
def test_side_scratch_follows_the_grid(hip_device, first, then):
    """The second stream is made by the first long pass, with scratch rows for
    the traversal grid of that time, after short passes have sized the first
    stream's rows for a larger one.  A later long pass with a larger grid than
    the second stream has seen gets rows for it: its frame, full of hits
    recorded in those rows, equals the oracle's."""
    sc = scenes.c1(width=256, height=144, spp=4, grid=97, instances=160)  # 147,456 paths
    for m in range(1, len(sc.materials)):
        sc.materials[m] = {"type": "glass", "eta": 1.5}
    small = scenes.c0(64, 64)
    L = K.lib()
    handles = []
    dev = A.init("hip", traceBlocksPerCU=64)  # a device of its own: no second stream yet
    try:
        def frame(scene, fmt=K.OSP_FB_RGBA32F):
            s = scenes.to_ospray(scene)
            fb = A.framebuffer(scene.width, scene.height, fmt, K.OSP_FB_COLOR | K.OSP_FB_ACCUM)
            handles.extend([fb, s.renderer, s.camera, s.world] + s.handles)
            A.render(fb, s.renderer, s.camera, s.world)
            return A.map_color(fb, scene.width, scene.height, fmt)

        frame(small)
        for blocks in (first, then):
            A.set_device_param(dev, "traceBlocksPerCU", blocks)
            L.ospDeviceCommit(dev)
            got = frame(sc)
    finally:
        for h in handles:
            h.release()
        L.ospSetCurrentDevice(hip_device)
        L.ospDeviceRelease(dev)
    ofb, _, _ = orc.render_scene(sc, frames=1, fmt=K.OSP_FB_RGBA32F, channels=K.OSP_FB_COLOR | K.OSP_FB_ACCUM)
    assert np.array_equal(got, ofb.channel(K.OSP_FB_COLOR))
