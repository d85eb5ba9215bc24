"""Passes of 2^17 paths or more run the shadow stages on a second stream,
shorter ones on one: around the line, with surfaces and with a volume, the
frame equals the one that overlapShadow false makes, bit for bit."""
import numpy as np
import pytest

from ospray_amd import api as A
from ospray_amd import capi as K
from ospray_amd import scenes

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
