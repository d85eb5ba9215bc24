"""How the traversal kernels deal out their queues changes only which rays
share a wave.  A queue of at least 64 entries per wave of the grid is taken
in 64-entry batches by whichever wave asks next; one of at most 4 entries per
wave is left to whole waves, a ray each; one in between (the last bounces of a
large frame) is spread as one batch of ceil(n / waves) entries per wave.  With
one traversal block per CU (512 waves on 256 CUs) the 36,864 rays of the
128x72, 4 spp frame's first bounce run batched, its later bounces spread and
its last ones by whole waves; with the default 12 (6,144 waves) the first
bounces are spread; with 64 every queue is left to whole waves.  Frames
rendered at 1, 64 and the default number of blocks per CU are equal bit for
bit, and equal to the oracle."""
import numpy as np
import pytest

from ospray_amd import api as A
from ospray_amd import capi as K
from ospray_amd import scenes
from oracle import orc

pytestmark = pytest.mark.gpu

W, H, SPP = 128, 72, 4
CH = K.OSP_FB_COLOR | K.OSP_FB_ACCUM | K.OSP_FB_DEPTH | K.OSP_FB_ID_PRIMITIVE | K.OSP_FB_ID_INSTANCE


def _scene():
    # all materials, the sun cone and four quad lights, instancing
    return scenes.c1(width=W, height=H, spp=SPP, grid=97, instances=40)


def _render(blocks_per_cu):
    L = K.lib()
    dev = L.ospGetCurrentDevice()
    if blocks_per_cu is not None:
        A.set_device_param(dev, "traceBlocksPerCU", blocks_per_cu)
        L.ospDeviceCommit(dev)
    try:
        A.check()
        sc = _scene()
        s = scenes.to_ospray(sc)
        fb = A.framebuffer(W, H, K.OSP_FB_RGBA32F, CH)
        A.render(fb, s.renderer, s.camera, s.world)
        return [A.map_color(fb, W, H, K.OSP_FB_RGBA32F)] + [A.map_channel(fb, c, W, H) for c in
                                                           (K.OSP_FB_DEPTH, K.OSP_FB_ID_PRIMITIVE,
                                                            K.OSP_FB_ID_INSTANCE)]
    finally:
        if blocks_per_cu is not None:
            A.set_device_param(dev, "traceBlocksPerCU", 12)
            L.ospDeviceCommit(dev)


def test_queue_batching_renders_the_same_frame(hip_device):
    base = _render(None)
    for bpc in (1, 64):
        other = _render(bpc)
        for k, (a, b) in enumerate(zip(base, other)):
            assert np.array_equal(a, b, equal_nan=True), (bpc, k)
    ofb, _, _ = orc.render_scene(_scene(), frames=1, fmt=K.OSP_FB_RGBA32F, channels=CH)
    assert np.array_equal(base[0], ofb.channel(K.OSP_FB_COLOR))
    for arr, ch in zip(base[1:], (K.OSP_FB_DEPTH, K.OSP_FB_ID_PRIMITIVE, K.OSP_FB_ID_INSTANCE)):
        assert np.array_equal(arr, ofb.channel(ch), equal_nan=True), ch


def _glass_scene():
    # every instance glass, so that shadow rays through them fill the
    # transparency queue: more than 64 entries per wave with one traversal
    # block per CU (512 waves), fewer than one per wave with 64
    sc = scenes.c1(width=256, height=144, spp=4, grid=97, instances=160)
    for i in range(1, len(sc.materials)):
        sc.materials[i] = {"type": "glass", "eta": 1.5}
    return sc


@pytest.mark.parametrize("bpc", [1, 12, 64])
def test_transparency_queue_of_any_length(hip_device, bpc):
    """Wave w of the transparency pass owns the entries from w * per on, in
    strides of waves * per: the frame equals the oracle's whatever the number
    of waves (no recorded hit is skipped or replayed twice)."""
    L = K.lib()
    dev = L.ospGetCurrentDevice()
    A.set_device_param(dev, "traceBlocksPerCU", bpc)
    L.ospDeviceCommit(dev)
    try:
        sc = _glass_scene()
        s = scenes.to_ospray(sc)
        fb = A.framebuffer(sc.width, sc.height, K.OSP_FB_RGBA32F, CH)
        A.render(fb, s.renderer, s.camera, s.world)
        got = A.map_color(fb, sc.width, sc.height, K.OSP_FB_RGBA32F)
    finally:
        A.set_device_param(dev, "traceBlocksPerCU", 12)
        L.ospDeviceCommit(dev)
    ofb, _, _ = orc.render_scene(sc, frames=1, fmt=K.OSP_FB_RGBA32F, channels=CH)
    assert np.array_equal(got, ofb.channel(K.OSP_FB_COLOR))


@pytest.mark.parametrize("depths", [(2, 30, 2), (0, 1, 40)])
def test_counters_follow_the_path_length(hip_device, depths):
    """Each bounce has counters of its own, sized for the longest path so
    far: frames of growing and shrinking path length, in one pass and in two
    (the smallest path budget, 64 MB, holds two samples of the larger frame),
    equal the oracle's."""
    L = K.lib()
    dev = L.ospGetCurrentDevice()
    for budget, w, h in ((16384, 24, 16), (64, 256, 192)):
        A.set_device_param(dev, "pathBudgetMB", budget)
        L.ospDeviceCommit(dev)
        try:
            for d in depths:
                sc = scenes.c0(w, h, spp=3, max_path_length=d)
                s = scenes.to_ospray(sc)
                fb = A.framebuffer(w, h, K.OSP_FB_RGBA32F, CH)
                A.render(fb, s.renderer, s.camera, s.world)
                ofb, _, _ = orc.render_scene(sc, frames=1, fmt=K.OSP_FB_RGBA32F, channels=CH)
                assert np.array_equal(A.map_color(fb, w, h, K.OSP_FB_RGBA32F), ofb.channel(K.OSP_FB_COLOR)), (budget, d)
        finally:
            A.set_device_param(dev, "pathBudgetMB", 16384)
            L.ospDeviceCommit(dev)
