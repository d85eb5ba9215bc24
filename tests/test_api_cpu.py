"""The C-ABI boundary on the CPU: exported symbols, module loading, the
object layer and error behaviour (ospray/api/API.cpp:45-66, 86-153;
ospray/common/OSPCommon.cpp:749-782; OSPCommon.h:126-133).  No GPU work is
launched here; commits that need device memory are not exercised."""
import ctypes as C
import os
import re
import subprocess

import pytest

from ospray_amd import capi as K

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared(header, macro):
    text = open(os.path.join(ROOT, "include", header)).read()
    return sorted(set(re.findall(macro + r"\s+[\w\s\*]+?\b(\w+)\s*\(", text)))


def _exports(lib):
    out = subprocess.run(["nm", "-D", "--defined-only", lib], capture_output=True, text=True, check=True).stdout
    return {line.split()[-1] for line in out.splitlines() if line.strip()}


def test_core_exports_every_declared_function():
    names = _declared("ospray/ospray.h", "OSPRAY_INTERFACE") + _declared("ospray/ospray_util.h", "OSPRAY_INTERFACE")
    assert len(names) == 77  # ospray.h (51) + ospray_util.h (26) of OSPRay 3.3
    exported = _exports(os.path.join(K.LIBDIR, "libospray.so"))
    missing = [n for n in names if n not in exported]
    assert not missing, missing


def test_module_exports_every_declared_function():
    names = (_declared("ospray/ospray_hip.h", "OSPRAY_INTERFACE") + _declared("ospray_hip/hip_pt.h", "HPT_API")
             + _declared("ospray_hip/hip_nrc.h", "HPT_API") + _declared("ospray_hip/hip_bvh.h", "HPT_API"))
    assert "hpt_extend" in names and "ospHipTraceRays" in names and "hpt_nrc_train" in names
    assert "hpt_bvh_build" in names and "ospHipGetWorldBuild" in names
    exported = _exports(os.path.join(K.LIBDIR, "libospray_module_hip.so"))
    missing = [n for n in names + ["ospray_module_init_hip"] if n not in exported]
    assert not missing, missing


def test_stage_entry_points_stay():
    """What a caller of the stage kernels was given stays, with its arguments."""
    text = " ".join(open(os.path.join(ROOT, "include", "ospray_hip", "hip_pt.h")).read().split())
    text += " ".join(open(os.path.join(ROOT, "include", "ospray_hip", "hip_bvh.h")).read().split())
    for decl in ("hpt_reset_counters(const HptPaths *P, int keepIndex, hipStream_t s)",
                 "hpt_reset_extension_counters(const HptPaths *P, int keepIndex, hipStream_t s)",
                 "hpt_reset_append_counters(const HptPaths *P, int keepIndex, hipStream_t s)",
                 "hpt_reset_shadow_counters(const HptPaths *P, hipStream_t s)",
                 "hpt_finish_pass(const HptFrame *F, const HptPaths *P, hipStream_t s)",
                 "hpt_fb_accumulate(const HptFrame *F, hipStream_t s)",
                 "hpt_color_convert(const float *color, int npix, int format, void *out, hipStream_t s)",
                 "hpt_bvh_relocate(void *dst, const void *src, size_t n, int32_t nodeOffset, uint32_t primOffset, "
                 "hipStream_t s)"):
        assert "HPT_API hipError_t " + decl + ";" in text, decl


def test_at_bounce_needs_counters_per_bounce():
    """hpt_at_bounce returns nothing that could say an error: without P->pass,
    or before the first bounce, P keeps the counters it has."""
    lib = C.CDLL(os.path.join(K.LIBDIR, "libospray_module_hip.so"), mode=C.RTLD_GLOBAL)
    state = (C.c_uint64 * 512)()  # no smaller than the path state
    lib.hpt_at_bounce(state, 3)
    assert not any(state)
    for i in range(len(state)):
        state[i] = 1 << 40
    lib.hpt_at_bounce(state, -1)
    assert all(v == 1 << 40 for v in state)
    lib.hpt_at_bounce(state, 1)  # the bounce's counters, its stages' and the next bounce's
    assert sum(v != 1 << 40 for v in state) == 3


def test_module_version_check():
    lib = C.CDLL(os.path.join(K.LIBDIR, "libospray_module_hip.so"), mode=C.RTLD_GLOBAL)
    init = lib.ospray_module_init_hip
    init.restype = C.c_int
    init.argtypes = [C.c_int16, C.c_int16, C.c_int16]
    assert init(2, 0, 0) == K.OSP_VERSION_MISMATCH
    assert init(3, 2, 0) == K.OSP_VERSION_MISMATCH
    assert init(3, 3, 0) == K.OSP_NO_ERROR


def _run(code):
    """Run a snippet in a fresh interpreter (the C API keeps global state)."""
    r = subprocess.run(["python3", "-c", code], capture_output=True, text=True, cwd=ROOT, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


def test_calls_without_device_fail_cleanly():
    out = _run(
        "from ospray_amd import capi as K\n"
        "L = K.lib()\n"
        "print(L.ospNewCamera(b'perspective') is None)\n"
        "print(L.ospGetVariance(None))\n"
        "print(L.ospLoadModule(b'doesnotexist'))\n"
        "print(L.ospNewDevice(b'nosuchdevice') is None)\n")
    lines = out.split()
    assert lines == ["True", "inf", str(K.OSP_UNKNOWN_ERROR), "True"]


def test_object_layer_and_errors():
    out = _run(
        "from ospray_amd import api as A, capi as K\n"
        "A.init('hip')\n"
        "L = K.lib()\n"
        "for kind, t in [('camera','perspective'), ('material','obj'), ('material','metal'), ('material','glass'),"
        " ('light','quad'), ('light','distant'), ('light','ambient')]:\n"
        "    A.new(kind, t, {})\n"
        "for kind, t in [('camera','orthographic'), ('renderer','scivis'), ('geometry','curve'), ('light','hdri')]:\n"
        "    try:\n"
        "        A.new(kind, t, {})\n"
        "        print('accepted', kind, t)\n"
        "    except A.OSPRayError as e:\n"
        "        print('rejected', 'Could not find' in str(e))\n"
        "A.new('material', 'obj', {'ks': (0.5, 0.5, 0.5), 'ns': 20.0})\n"
        "print('ks accepted')\n"
        "cam = A.new('camera', 'perspective', {'fovy': 30.0})\n"
        "L.ospRelease(cam.h)\n"
        "print('property', L.ospDeviceGetProperty(L.ospGetCurrentDevice(), 1))\n")
    lines = out.strip().splitlines()
    assert lines[:4] == ["rejected True"] * 4
    assert lines[4] == "ks accepted"
    assert lines[5] == "property 3"


def test_framebuffer_variance_requires_accum():
    # ospNewFrameBuffer drops VARIANCE without ACCUM (API.cpp:568-582); the
    # check happens before any device call, so it is visible in the handle's
    # channel mask only through behaviour: here just that creation of a
    # framebuffer of invalid size fails with an error.
    out = _run(
        "from ospray_amd import api as A, capi as K\n"
        "A.init('hip')\n"
        "h = K.lib().ospNewFrameBuffer(0, 10, K.OSP_FB_RGBA8, K.OSP_FB_COLOR)\n"
        "print(h is None)\n"
        "try:\n"
        "    A.check()\n"
        "except A.OSPRayError as e:\n"
        "    print('invalid size' in str(e))\n")
    assert out.split() == ["True", "True"]


def test_c_application_compiles_against_headers(tmp_path):
    """An application written only against include/ospray/*.h compiles and
    links against libospray.so (the drop-in boundary)."""
    src = os.path.join(ROOT, "tests", "apps", "pathtracer_app.c")
    exe = str(tmp_path / "app")
    subprocess.run(["gcc", "-std=c99", "-Wall", "-Werror", "-o", exe, src, f"-I{ROOT}/include", f"-L{K.LIBDIR}",
                    "-lospray", f"-Wl,-rpath,{K.LIBDIR}", "-lm"], check=True)
    assert os.path.exists(exe)


@pytest.mark.parametrize("std", ["c++11", "c++17"])
def test_cpp_application_compiles_against_wrapper(tmp_path, std):
    """The C++ wrapper (include/ospray/ospray_cpp.h) compiles warning-free
    in an application and links against libospray.so."""
    src = os.path.join(ROOT, "tests", "apps", "pathtracer_cpp_app.cpp")
    exe = str(tmp_path / "app")
    subprocess.run(["g++", f"-std={std}", "-Wall", "-Wextra", "-Werror", "-o", exe, src, f"-I{ROOT}/include",
                    f"-L{K.LIBDIR}", "-lospray", f"-Wl,-rpath,{K.LIBDIR}"], check=True)
    assert os.path.exists(exe)


_WRAPPER_CHECKS = r"""
#include <array>
#include <vector>
#include "ospray/ospray_cpp.h"
#include "ospray/ospray_cpp/ext/glm.h"
#include "ospray/ospray_cpp/ext/rkcommon.h"
using namespace ospray;
static_assert(OSPTypeFor<float>::value == OSP_FLOAT, "");
static_assert(OSPTypeFor<const char *>::value == OSP_STRING, "");
static_assert(OSPTypeFor<OSPFrameBufferFormat>::value == OSP_UINT, "");
static_assert(OSPTypeFor<cpp::Camera>::value == OSP_CAMERA, "");
static_assert(OSPTypeFor<cpp::GeometricModel>::value == OSP_GEOMETRIC_MODEL, "");
static_assert(OSPTypeFor<cpp::CopiedData>::value == OSP_DATA, "");
static_assert(OSPTypeFor<cpp::MovedData>::value == OSP_DATA, "");
static_assert(OSPTypeFor<glm::vec3>::value == OSP_VEC3F, "");
static_assert(OSPTypeFor<glm::mat4x3>::value == OSP_AFFINE3F, "");
static_assert(OSPTypeFor<rkcommon::math::vec3ul>::value == OSP_VEC3UL, "");
static_assert(OSPTypeFor<rkcommon::math::box1f>::value == OSP_BOX1F, "");
static_assert(OSPTypeFor<rkcommon::math::affine3f>::value == OSP_AFFINE3F, "");
static_assert(OSPTypeFor<std::vector<int>>::value == OSP_UNKNOWN, "");
static_assert(sizeof(cpp::World) == sizeof(OSPWorld) && sizeof(cpp::SharedData) == sizeof(OSPData), "");
OSPTYPEFOR_DEFINITION(glm::vec3);
void use(const rkcommon::math::vec3ul &dims, const std::array<float, 8> &a, const float *p)
{
  cpp::SharedData d3(p, dims);             // 3D dimensions from a registered vector
  cpp::CopiedData c(a);                    // std::array
  cpp::Volume v("structuredRegular");
  v.setParam("data", d3);
  v.setParam("gridSpacing", glm::vec3{1.f, 1.f, 1.f});
  v.setParam("name", std::string("v"));
  v.removeParam("name");
  cpp::Device dev("hip");
  dev.setParam("numThreads", 4);
  dev.setParam("logOutput", "cerr");
}
"""


def test_cpp_wrapper_type_registry(tmp_path):
    """OSPTypeFor of the wrapper classes, the enums and the glm / rkcommon
    registrations (ext/glm.h, ext/rkcommon.h); glm and rkcommon are not in
    this image, so minimal types with their names stand in for them, enough
    to instantiate the registrations."""
    for sub, names in (("glm", ["vec2.hpp", "vec3.hpp", "vec4.hpp", "mat2x2.hpp", "mat3x2.hpp", "mat3x3.hpp",
                                "mat4x3.hpp"]), ("rkcommon/math", ["AffineSpace.h", "box.h"])):
        d = tmp_path / sub
        d.mkdir(parents=True)
        for n in names:
            # distinct text: gcc's #pragma once takes identical files for one
            (d / n).write_text(f"#pragma once\n// {sub}/{n}\n#include \"types.h\"\n")
    (tmp_path / "glm" / "types.h").write_text(
        "#pragma once\nnamespace glm {\n" + "".join(
            f"struct {t} {{ float v[{n}]; }};\n" for t, n in
            (("vec2", 2), ("vec3", 3), ("vec4", 4), ("ivec2", 2), ("ivec3", 3), ("ivec4", 4), ("uvec2", 2),
             ("uvec3", 3), ("uvec4", 4), ("mat2x2", 4), ("mat3x3", 9), ("mat3x2", 6), ("mat4x3", 12))) + "}\n")
    rk = ["vec2uc", "vec3uc", "vec4uc", "vec2c", "vec3c", "vec4c", "vec2us", "vec3us", "vec4us", "vec2s", "vec3s",
          "vec4s", "vec2i", "vec3i", "vec4i", "vec2ui", "vec3ui", "vec4ui", "vec2l", "vec3l", "vec4l", "vec2ul",
          "vec4ul", "vec2f", "vec3f", "vec4f", "vec2d", "vec3d", "vec4d", "box1i", "box2i", "box3i", "box4i",
          "box1f", "box2f", "box3f", "box4f", "linear2f", "linear3f", "affine2f", "affine3f", "quatf"]
    (tmp_path / "rkcommon" / "math" / "types.h").write_text(
        "#pragma once\n#include <cstdint>\nnamespace rkcommon { namespace math {\n"
        "struct vec3ul { uint64_t v[3]; uint64_t operator[](int i) const { return v[i]; } };\n"
        + "".join(f"struct {t} {{ float v[4]; }};\n" for t in rk) + "} }\n")
    src = tmp_path / "checks.cpp"
    src.write_text(_WRAPPER_CHECKS)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-c", "-o", str(tmp_path / "checks.o"),
                    str(src), f"-I{ROOT}/include", f"-I{tmp_path}"], check=True)
