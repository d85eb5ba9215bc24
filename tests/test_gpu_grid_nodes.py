"""The traversal's nodes hold their children's boxes on an 8-bit grid, rounded
outwards: whatever the boxes' sizes (flat, far apart in size, tiny, far from
the origin) and however many slots a node uses, the closest hits are the
oracle's bit for bit, since the boxes only cull."""
import numpy as np
import pytest

from ospray_amd import api as A
from ospray_amd import capi as K
from ospray_amd import scenes
from oracle import orc

pytestmark = pytest.mark.gpu


def _triangles(shape, n, scale, offset, rng):
    c = rng.uniform(-1, 1, (n, 1, 3))
    size = {"cloud": 0.3, "flat": 0.3, "sizes": 1.0}[shape]
    if shape == "sizes":  # over four orders of magnitude within one tree
        size = 10.0 ** rng.uniform(-4, 0, (n, 1, 1))
    v = c + size * rng.uniform(-1, 1, (n, 3, 3))
    if shape == "flat":  # every box without extent along y
        v[:, :, 1] = 0.25
    return (scale * v + np.array(offset)).reshape(-1, 3).astype(np.float32)


def _rays(v, rng, n=4000):
    lo, hi = v.min(0), v.max(0)
    mid, ext = 0.5 * (lo + hi), float((hi - lo).max())
    o = mid + ext * rng.uniform(-1.5, 1.5, (n, 3))
    t = v[rng.integers(0, len(v), n)] + 0.05 * ext * rng.normal(size=(n, 3))
    d = t - o
    axis = rng.integers(0, 3, n // 4)  # a quarter parallel to an axis
    d[: n // 4] = np.eye(3)[axis] * rng.choice([-1.0, 1.0], (n // 4, 1))
    o[: n // 4] = t[: n // 4] - 2.0 * ext * d[: n // 4]
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return np.concatenate([o, d, np.zeros((n, 1)), np.full((n, 1), np.inf)], 1).astype(np.float32)


@pytest.mark.parametrize("host", [True, False])
@pytest.mark.parametrize("shape,n,scale,offset", [
    ("cloud", 1, 1.0, (0, 0, 0)), ("cloud", 2, 1.0, (0, 0, 0)), ("cloud", 3, 1.0, (0, 0, 0)),
    ("cloud", 5, 1.0, (0, 0, 0)), ("cloud", 9, 1e-3, (0, 0, 0)), ("cloud", 700, 1.0, (40, -30, 90)),
    ("flat", 300, 1.0, (0, 0, 0)), ("flat", 2, 100.0, (0, 7, 0)), ("sizes", 600, 1.0, (0, 0, 0)),
    ("sizes", 600, 50.0, (0, 500, 0))])
def test_hits_equal_the_oracle(hip_device, shape, n, scale, offset, host):
    rng = np.random.default_rng(n)
    v = _triangles(shape, n, scale, offset, rng)
    geoms = [scenes.Geometry("triangles", vertex=v, index=np.arange(3 * n, dtype=np.uint32).reshape(-1, 3))]
    insts = [scenes.Instance(0), scenes.Instance(0, xfm=(0.5, 0, 0, 0, -0.7, 0, 0.1, 0, 0.6, 0.3 * scale, 0, 0))]
    sc = scenes.Scene("grid", 8, 8, geoms, [scenes.Model(0, 0)], [[0]], insts, [{"type": "obj"}],
                      [{"type": "ambient"}], {"position": (0, 0, -1), "direction": (0, 0, 1)}, {"pixelSamples": 1})
    dev = K.lib().ospGetCurrentDevice()
    A.set_device_param(dev, "hostBvh", host)
    K.lib().ospDeviceCommit(dev)
    try:
        s = scenes.to_ospray(sc)
    finally:
        A.set_device_param(dev, "hostBvh", True)
        K.lib().ospDeviceCommit(dev)
    rays = _rays(v, rng)
    tuv, ids, _ = A.trace_rays(s.world, rays)
    otuv, oids, _ = orc.OracleScene(sc).intersect(rays)
    assert np.array_equal(ids, oids) and np.array_equal(tuv, otuv)
    assert (ids[:, 0] != 0xFFFFFFFF).any()


@pytest.mark.parametrize("n", [1, 2, 3])
def test_unused_slots_are_not_entered(hip_device, n):
    """A node of one to three children leaves the others' slots unused: rays
    into the node's own corners, the lowest ones among them, test no more
    primitives than it has."""
    rng = np.random.default_rng(7 + n)
    v = rng.uniform(0.1, 0.9, (n, 3, 3)).astype(np.float32)
    v[0, 0], v[0, 1], v[0, 2] = (0, 0, 0), (1, 1, 1), (0, 1, 0.5)  # the node's box: the unit cube
    sc = scenes.Scene("corner", 8, 8, [scenes.Geometry("triangles", vertex=v.reshape(-1, 3),
                                                       index=np.arange(3 * n, dtype=np.uint32).reshape(-1, 3))],
                      [scenes.Model(0, 0)], [[0]], [scenes.Instance(0)], [{"type": "obj"}], [{"type": "ambient"}],
                      {"position": (0, 0, -1), "direction": (0, 0, 1)}, {"pixelSamples": 1})
    s = scenes.to_ospray(sc)
    corners = np.array([[x, y, z] for x in (0, 1) for y in (0, 1) for z in (0, 1)], np.float64)
    rays = []
    for c in corners:
        for _ in range(16):
            d = rng.normal(size=3)
            d /= np.linalg.norm(d)
            rays.append(np.concatenate([c - 3 * d, d, [0, np.inf]]))
    rays = np.array(rays, np.float32)
    tuv, ids, (nodes, prims) = A.trace_rays(s.world, rays)
    otuv, oids, _ = orc.OracleScene(sc).intersect(rays)
    assert np.array_equal(ids, oids) and np.array_equal(tuv, otuv)
    assert prims <= n * len(rays), prims


def _visits(v, rays, xfms):
    n = len(v) // 3
    sc = scenes.Scene("scales", 8, 8, [scenes.Geometry("triangles", vertex=v,
                                                       index=np.arange(3 * n, dtype=np.uint32).reshape(-1, 3))],
                      [scenes.Model(0, 0)], [[0]], [scenes.Instance(0, xfm=x) for x in xfms], [{"type": "obj"}],
                      [{"type": "ambient"}], {"position": (0, 0, -1), "direction": (0, 0, 1)}, {"pixelSamples": 1})
    s = scenes.to_ospray(sc)
    tuv, ids, visits = A.trace_rays(s.world, rays)
    otuv, oids, _ = orc.OracleScene(sc).intersect(rays)
    assert np.array_equal(ids, oids) and np.array_equal(tuv, otuv)
    assert (ids[:, 0] != 0xFFFFFFFF).any()
    return np.array(visits, np.float64)


ID = (1, 0, 0, 0, 1, 0, 0, 0, 1)


def test_culling_is_local(hip_device):
    """What a ray visits next to small detail depends neither on objects far
    away, in the world or in the same geometry, nor on the distance to the
    origin of the coordinates: the padding of a box is made of the box's own
    size and its distance to the ray's origin."""
    rng = np.random.default_rng(5)
    # 2,000 triangles of 0.1 in a cube of 8, on a grid of 1/64, so that they
    # can be moved by 2^17 without a rounding
    c = rng.uniform(-4, 4, (2000, 1, 3))
    v = (np.round(64 * (c + 0.1 * rng.uniform(-1, 1, (2000, 3, 3)))) / 64).reshape(-1, 3).astype(np.float32)
    # (rays along an axis through the grid's points would run in the faces of
    # the oracle's boxes, which miss what lies in the face)
    rays = _rays(v, rng)[1000:]
    rays[:, :3] = np.round(64 * rays[:, :3]) / 64
    base = _visits(v, rays, [ID + (0, 0, 0)])
    # an instance far away: the same rays miss it at the root
    far = _visits(v, rays, [ID + (0, 0, 0), ID + (1e6, 0, 0)])
    assert np.all(far <= 1.02 * base + len(rays) * np.array([0.1, 0.1])), (far, base)
    # one triangle far away: a node or two more above the others, and those
    # the root's coarse grid lets a ray into
    w = np.concatenate([v, v[:3] + np.float32([1e6, 0, 0])])
    one = _visits(w, rays, [ID + (0, 0, 0)])
    assert np.all(one <= 1.1 * base + len(rays) * np.array([3, 0.2])), (one, base)
    # everything moved away from the origin
    moved = rays.copy()
    moved[:, :3] += np.float32(2 ** 17)
    away = _visits(v + np.float32(2 ** 17), moved, [ID + (0, 0, 0)])
    assert np.all(away <= 1.1 * base + len(rays) * 0.1), (away, base)
