"""The BVH's packed nodes (f16 planes, rounded outwards from a node's own
origin and scale) lose no hit: against the oracle's exhaustive instance loop,
from tiny to huge scenes, near and far from the world's origin, still and
moving, with sizes far apart in one node."""
import numpy as np
import pytest

from oracle import ora
from psychopath_cpp_amd import abi
from psychopath_cpp_amd.scene import Assembly, Camera, Scene, Sphere, look_at, translate
from tests.cpu_build import hostbuild


def _field(scale, offset, moving, n=300, seed=4):
    rng = np.random.default_rng(seed)
    root = Assembly()
    o = np.asarray(offset, np.float64) * scale
    eye = o + np.array([0.0, -30.0, 4.0]) * scale
    sc = Scene(Camera([look_at(eye, o)], [0.7]), root)
    sc.add_surface_shader("s", abi.PSY_SHADER_LAMBERT, (0.5, 0.5, 0.5))
    for i in range(n):
        c = o + rng.uniform(-8, 8, 3) * scale
        r = float(np.exp(rng.uniform(np.log(0.01), np.log(2.0)))) * scale
        root.add_object(f"o{i}", Sphere((0.0, 0.0, 0.0), r))
        xs = [translate(*c)]
        if moving:
            xs.append(translate(*(c + rng.uniform(-3, 3, 3) * scale)))
        root.create_object_instance(f"o{i}", xs, "s")
    return sc


@pytest.mark.parametrize("moving", [False, True])
@pytest.mark.parametrize("scale,offset", [(1.0, (0, 0, 0)), (1e-4, (0, 0, 0)), (1e5, (0, 0, 0)), (1e12, (0, 0, 0)),
                                          (1.0, (500, -300, 100))])
def test_packed_nodes_lose_no_hit(scale, offset, moving):
    sc = _field(scale, offset, moving)
    o = ora.OracleScene(sc)
    w, _ = o.camera_rays(72, 48, 1, 2)
    hb = hostbuild.trace(sc, ora.planes_from_wrays(w), world=True, dice_depth=0)
    inter = o.trace(w, threads=8, chunk=4096, brute=True)
    hit = hb["inst"] != 0xFFFFFFFF
    assert hit.sum() > 500
    assert np.array_equal(hit, inter["hit"] != 0)
    # the oracle's sphere test runs in single precision far from the origin as well: the same instance, and the same
    # distance to that precision
    t = inter["t"][hit]
    assert np.mean(np.abs(hb["t"][hit] - t) <= 1e-5 * np.abs(t)) >= 0.999


def test_rays_out_of_the_nodes_range_take_the_second_pass():
    """Directions so flat that slab distances could overflow are not tested
    against packed nodes."""
    sc = _field(1.0, (0, 0, 0), False)
    o = ora.OracleScene(sc)
    w, _ = o.camera_rays(24, 16, 1, 2)
    w["d"][::2, 0] = 1e-37
    w["d"][1::2, 0] = 0.0
    hb = hostbuild.trace(sc, ora.planes_from_wrays(w), world=True, dice_depth=0)
    assert hb["retraced"] == len(w)
    inter = o.trace(w, threads=8, chunk=4096, brute=True)
    assert np.array_equal(hb["inst"] != 0xFFFFFFFF, inter["hit"] != 0)
