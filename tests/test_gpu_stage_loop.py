"""The stage kernels' C ABI (include/ospray_hip/hip_pt.h) called by a program
of its own (tests/apps/stage_loop.cpp) instead of the device: with a block of
counters for each bounce, and with the same counters for every bounce, cleared
whole or in parts, a frame of two passes equals the device's bit for bit."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from ospray_amd import api as A
from ospray_amd import capi as K
from ospray_amd import scenes

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def stage_loop(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stage") / "stage_loop.so")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", f"-I{ROOT}/include",
                    f"-I{ROOT}/ospray_amd/csrc/hip", f"-I{rocm}/include", "-o", so,
                    os.path.join(ROOT, "tests", "apps", "stage_loop.cpp"), f"-L{K.LIBDIR}", "-l:libospray_module_hip.so",
                    f"-Wl,-rpath,{K.LIBDIR}", f"-L{rocm}/lib", "-lamdhip64"], check=True)
    lib = C.CDLL(so)
    lib.begin_pass.argtypes = [C.c_void_p, C.c_int]
    f = lib.stage_loop
    f.restype = C.c_int
    f.argtypes = [C.c_void_p] + [C.c_int] * 5 + [C.c_float, C.c_void_p, C.c_int, C.c_int, C.c_void_p, C.c_void_p]
    return lib


def _scene():
    # the box of test_gpu_nrc.py's kind: materials of three kinds, glass among
    # them (the transparency pass), a quad light and an ambient one
    sc = scenes.c0(72, 40, 4, 6)
    for i, m in enumerate(({"type": "glass", "eta": 1.5}, {"type": "metal", "roughness": 0.2})):
        sc.materials.append(m)
        sc.models[i + 1].material = len(sc.materials) - 1
    sc.camera = {"position": (0.0, 1.0, -12.0), "direction": (0.0, 0.0, 1.0), "up": (0.0, 1.0, 0.0), "fovy": 50.0,
                 "aspect": 72 / 40}
    return sc


@pytest.mark.parametrize("counters", [0, 1, 2])
def test_frame_equals_the_device(hip_device, stage_loop, counters):
    sc = _scene()
    w, h, spp, depth = sc.width, sc.height, 4, 6
    s = scenes.to_ospray(sc, {"pixelSamples": spp, "maxPathLength": depth, "pixelFilter": A.UInt(K.OSP_PIXELFILTER_POINT)})
    want = {}
    for fmt in (K.OSP_FB_RGBA32F, K.OSP_FB_SRGBA):
        fb = A.framebuffer(w, h, fmt, K.OSP_FB_COLOR | K.OSP_FB_ACCUM)
        A.render(fb, s.renderer, s.camera, s.world)
        want[fmt] = A.map_color(fb, w, h, fmt)
    mod = C.CDLL(os.path.join(K.LIBDIR, "libospray_module_hip.so"))
    mod.ospHipGetWorldLaunchScene.restype = C.c_void_p
    mod.ospHipGetWorldLaunchScene.argtypes = [C.c_void_p]
    scene = mod.ospHipGetWorldLaunchScene(s.world.h)
    color, words = np.zeros((h, w, 4), np.float32), np.zeros((h, w), np.uint32)
    pos = np.array(sc.camera["position"], np.float32)
    rc = stage_loop.stage_loop(scene, w, h, spp, 2, depth, sc.camera["fovy"], pos.ctypes.data, counters, 64, color.ctypes.data,
                    words.ctypes.data)
    assert rc == 0
    assert want[K.OSP_FB_RGBA32F][..., :3].any()
    # (mapping a float colour clamps it at 0)
    mapped = np.maximum(color, np.float32(0))
    mapped[..., 3] = np.minimum(mapped[..., 3], np.float32(1))
    assert np.array_equal(mapped, want[K.OSP_FB_RGBA32F])
    assert np.array_equal(words.view(np.uint8).reshape(h, w, 4), want[K.OSP_FB_SRGBA])


@pytest.mark.parametrize("bounces", [0, 20, 7895200])
def test_counters_of_any_path_length(hip_device, stage_loop, bounces):
    """hpt_begin_pass clears hpt_counter_bytes(bounces) bytes, 17 GB (more than
    2^32 words) of them too."""
    torch = pytest.importorskip("torch")
    size = C.CDLL(os.path.join(K.LIBDIR, "libospray_module_hip.so")).hpt_counter_bytes
    size.restype = C.c_size_t
    size.argtypes = [C.c_int]
    words = size(bounces) // 4
    assert (words > 2 ** 32) == (bounces > 20)
    t = torch.ones(words + 64, dtype=torch.int32, device="cuda")
    assert stage_loop.begin_pass(t.data_ptr(), bounces) == 0
    torch.cuda.synchronize()
    edge = min(words, 1 << 22)
    assert not t[:edge].any() and not t[words - edge:words].any()
    assert t[words:].all()
    del t
    torch.cuda.empty_cache()


def test_relocated_nodes(hip_device):
    """hpt_bvh_relocate: nodes as the builders write them (six float4 of boxes,
    four child references, four words of padding), inner references moved by
    nodes, leaf references by primitives, unused slots (a box at +inf) as they are."""
    torch = pytest.importorskip("torch")
    mod = C.CDLL(os.path.join(K.LIBDIR, "libospray_module_hip.so"))
    mod.hpt_bvh_relocate.restype = C.c_int
    mod.hpt_bvh_relocate.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int32, C.c_uint32, C.c_void_p]
    rng = np.random.default_rng(3)
    n = 300
    boxes = rng.uniform(-1, 1, (n, 6, 4)).astype(np.float32)
    used = rng.uniform(size=(n, 4)) < 0.8
    boxes[np.broadcast_to(~used[:, None, :], boxes.shape)] = np.inf
    first, count = rng.integers(0, 1000, (n, 4)), rng.integers(0, 8, (n, 4))
    inner = rng.uniform(size=(n, 4)) < 0.5
    child = np.where(inner, first, ~(first << 3 | count)).astype(np.int32)
    want = np.where(used, np.where(inner, first + 77, ~((first + 123) << 3 | count)), child).astype(np.int32)
    words = np.concatenate([boxes.reshape(n, 24).view(np.int32), child, np.zeros((n, 4), np.int32)], 1)
    src = torch.tensor(words, device="cuda")
    dst = torch.zeros_like(src)
    assert mod.hpt_bvh_relocate(dst.data_ptr(), src.data_ptr(), n, 77, 123, None) == 0
    torch.cuda.synchronize()
    got = dst.cpu().numpy()
    words[:, 24:28] = want
    assert np.array_equal(got, words)
