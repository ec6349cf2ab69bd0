"""The traversal's packed box test on the CPU: tests/packed_check.cpp packs a scene's nodes with the code of
vulkanexp_amd/csrc/packed_node.hpp and traces rays through them with the kernels' FP32 operations.  Every
ray finds the nearest of all triangles, and it visits about as many nodes as with FP32 boxes: a plane is
rounded outward by at most one step of a 1024th of the node's extent, so a quarter more visits is a generous
bound (a box test that an axis no longer takes part in costs a multiple)."""
import dataclasses
import os
import subprocess

import numpy as np
import pytest

from vulkanexp_amd import scenes

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "vulkanexp_amd", "csrc")


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("packed") / "packed_check")
    cmd = ["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", out, os.path.join(ROOT, "tests", "packed_check.cpp"),
           os.path.join(CSRC, "bvh.cpp"), os.path.join(CSRC, "scene_io.cpp"), "-I" + os.path.join(ROOT, "include")]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    return out


def _scaled(scene, scale):
    v = scene.vertices.copy()
    v["pos"] = (v["pos"].astype(np.float64) * scale).astype(np.float32)
    return dataclasses.replace(scene, vertices=v)


def _beyond():
    """A room's boxes under a triangle too large for a node's grid."""
    sb = scenes.SceneBuilder()
    rng = np.random.Generator(np.random.PCG64(3))
    m = sb.add_material((0.5, 0.5, 0.5))
    for _ in range(40):
        lo = rng.uniform(0.0, 10.0, 3)
        p, n, t = scenes.box_mesh(lo, lo + rng.uniform(0.01, 2.0, 3))
        sb.add_instance(sb.add_mesh(p, n, t, m))
    p = np.array([[-2e37, 11.0, -2e37], [2e37, 11.0, -2e37], [0.0, 11.0, 2e37]], np.float32)
    sb.add_instance(sb.add_mesh(p, np.tile(np.float32([0, -1, 0]), (3, 1)), np.array([[0, 1, 2]]), m))
    return sb.build((0, 0, 0), (12, 12, 12))


SCENES = {
    "room": lambda: scenes.config_small(seed=1)[0],
    "clustered": lambda: scenes.clustered_scene(seed=5, n_instances=24),
    "room_1e-3": lambda: _scaled(scenes.config_small(seed=1)[0], 1e-3),
    "room_1e6": lambda: _scaled(scenes.config_small(seed=1)[0], 1e6),
    "room_1e14": lambda: _scaled(scenes.config_small(seed=1)[0], 1e14),
    "room_beyond": _beyond,
    "room_1e19": lambda: _scaled(scenes.config_small(seed=1)[0], 1e19),
}


def _trace(checker, tmp_path, scene, mode, rays, reach=1e30):
    path = str(tmp_path / "s.scene")
    scenes.save(scene, path)
    r = subprocess.run([checker, path, mode, str(rays), "23", str(reach)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    print(mode, r.stdout.strip())
    n, hits, bad, packed, fp32, most = r.stdout.split()
    return int(n), int(hits), int(bad), float(packed), float(fp32), int(most)


@pytest.mark.parametrize("mode", ["generic", "axis", "plane", "tiny"])
@pytest.mark.parametrize("name", sorted(SCENES))
def test_directions_with_components_near_zero(checker, tmp_path, name, mode):
    n, hits, bad, packed, fp32, most = _trace(checker, tmp_path, SCENES[name](), mode, 400 if name == "clustered" else 2000,
                                                12.0 if name == "room_beyond" else 1e30)
    assert hits > 0.1 * n
    assert bad == 0
    if name not in ("room_1e19", "room_beyond"):  # too large for bounded reciprocals: boxes are kept, and hits
        assert packed <= 1.25 * fp32


@pytest.mark.parametrize("mode", ["none", "infinite"])
@pytest.mark.parametrize("name", ["room", "clustered"])
def test_rays_that_hit_nothing_end_early(checker, tmp_path, name, mode):
    n, hits, bad, packed, fp32, most = _trace(checker, tmp_path, SCENES[name](), mode, 400)
    assert hits == 0 and bad == 0
    assert packed <= 1.25 * fp32


def _details(size):
    """A 200 m ground and details on it, each of seven triangles of extent `size`."""
    sb = scenes.SceneBuilder()
    rng = np.random.Generator(np.random.PCG64(8))
    m = sb.add_material((0.5, 0.5, 0.5))
    quad = np.array([[-100, 0, -100], [100, 0, -100], [100, 0, 100], [-100, 0, 100]], np.float32)
    sb.add_instance(sb.add_mesh(quad, np.tile(np.float32([0, 1, 0]), (4, 1)), np.array([[0, 1, 2], [0, 2, 3]]), m))
    tri = (rng.uniform(0.0, size, (21, 3)) + [0, 2 * size, 0]).astype(np.float32)
    mesh = sb.add_mesh(tri, np.tile(np.float32([0, 1, 0]), (21, 1)), np.arange(21).reshape(7, 3), m)
    for k in range(40):  # near the coordinates' origin, where small differences are exact
        sb.add_instance(mesh, np.array([[1, 0, 0, k % 8 * 8 * size], [0, 1, 0, 0], [0, 0, 1, k // 8 * 8 * size]], np.float32))
    return sb.build((-100, 0, -100), (100, 1, 100))


@pytest.mark.parametrize("size,reach", [(1e-4, 1e5), (1e-6, 1e4), (1e-3, 1e6), (1e-3, 1e2), (1e-5, 1e9), (1.0, 1e4)])
def test_small_details_from_far_away(checker, tmp_path, size, reach):
    """Rays from 1e4 to 1e14 detail sizes away, past details that have fewer than four children in a node."""
    n, hits, bad, packed, fp32, most = _trace(checker, tmp_path, _details(size), "far", 4000, reach)
    assert hits > 0.3 * n
    assert bad == 0
