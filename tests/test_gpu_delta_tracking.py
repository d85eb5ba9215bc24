"""Delta tracking at the edges of its macrocell walk (cells of 16 voxels):
grids of one cell, of a cell and a voxel, and a flat one, thin (nearly no
tentative collision) and dense (many in a cell), seen along an axis so that
rays have steps of zero: equal to the oracle bit for bit."""
import numpy as np
import pytest

from ospray_amd import api as A
from ospray_amd import capi as K
from ospray_amd import scenes
from test_gpu_parity import _add_volume_instance, _render_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("density", [0.05, 60.0])
@pytest.mark.parametrize("dims", [(2, 2, 2), (17, 16, 18), (33, 2, 50)])
def test_frames_equal_the_oracle(hip_device, dims, density):
    rng = np.random.default_rng(dims[0])
    vol = scenes.Volume(rng.random(dims).astype(np.float32), rng.uniform(0.4, 1.0, (4, 3)).astype(np.float32),
                        np.array([0.0, 0.3, 0.0, 0.5], np.float32), origin=(-1.0, -1.0, -1.0),
                        spacing=tuple(2.0 / (d - 1) for d in dims[::-1]), tf_range=(0.1, 0.9), density_scale=density,
                        anisotropy=0.2, user_id=None)
    sc = scenes.c0(33, 33, spp=2, max_path_length=4)
    sc.camera = dict(sc.camera, position=(0.0, 0.0, -12.0), direction=(0.0, 0.0, 1.0), up=(0.0, 1.0, 0.0), aspect=1.0)
    _add_volume_instance(sc, vol, (3, 0, 0, 0, 3, 0, 0, 0, 3, 0.0, 0.0, 0.0))
    s, fb, ofb, _, _ = _render_both(sc, frames=1)
    col = A.map_color(fb, sc.width, sc.height, K.OSP_FB_RGBA32F)
    assert np.array_equal(col, ofb.channel(K.OSP_FB_COLOR))
