"""The traversal's packed nodes (planes as small integers on a per-node grid): closest hits equal the
oracle's brute-force scan bit for bit, and any-hit decisions agree, where the grid or the distances
lose the most: tiny and large scenes, scenes far from the coordinates' origin, a node that holds a
huge triangle beside small ones, one too large for the grid, and ray origins far outside."""
import dataclasses

import numpy as np
import pytest

from oracle import py as orc
from vulkanexp_amd import scenes

pytestmark = pytest.mark.gpu


def _scene(scale, offset, big):
    sb = scenes.SceneBuilder()
    rng = np.random.Generator(np.random.PCG64(3))
    m = sb.add_material((0.5, 0.5, 0.5))
    for _ in range(40):
        lo = rng.uniform(0.0, 10.0, 3)
        p, n, t = scenes.box_mesh(lo, lo + rng.uniform(0.01, 2.0, 3))
        sb.add_instance(sb.add_mesh(p, n, t, m))
    if big:
        p = np.array([[-big, 11.0, -big], [big, 11.0, -big], [0.0, 11.0, big]], np.float32)
        sb.add_instance(sb.add_mesh(p, np.tile(np.float32([0, -1, 0]), (3, 1)), np.array([[0, 1, 2]]), m))
    s = sb.build((0, 0, 0), (12, 12, 12))
    v = s.vertices.copy()
    v["pos"] = (v["pos"].astype(np.float64) * scale + offset).astype(np.float32)
    return dataclasses.replace(s, vertices=v)


def _rays(scale, offset, n=6000):
    rng = np.random.Generator(np.random.PCG64(4))
    o = rng.uniform(-1.0, 13.0, (n, 3))
    far = rng.random(n) < 0.3
    o[far] = 6.0 + 1000.0 * rng.normal(size=(int(far.sum()), 3))
    at = rng.uniform(0.0, 12.0, (n, 3))
    d = at - o
    axis = rng.random(n) < 0.2   # along a coordinate axis, the other components +-0
    k = rng.integers(0, 3, n)
    flat = np.where(rng.random((n, 3)) < 0.5, 0.0, -0.0)
    flat[np.arange(n), k] = np.where(rng.random(n) < 0.5, 1.0, -1.0)
    d = np.where(axis[:, None], flat, d / np.linalg.norm(d, axis=1, keepdims=True))
    r = np.zeros((n, 8), np.float32)
    r[:, :3], r[:, 4:7], r[:, 7] = o * scale + offset, d, 1e5 * scale
    return r


@pytest.mark.parametrize("scale,offset,big", [(1.0, 0.0, 0.0), (1e-3, 0.0, 0.0), (1e4, 0.0, 0.0), (1.0, 3e3, 0.0),
                                              (1e-2, -40.0, 0.0), (1.0, 0.0, 1e6), (1.0, 0.0, 2e37)],
                         ids=["unit", "tiny", "large", "far", "tiny-far", "huge-triangle", "beyond-the-grid"])
def test_packed_nodes_keep_every_hit(scale, offset, big):
    from test_gpu_parity import _compare_hits, _gpu_trace, _make
    scene, rays = _scene(scale, offset, big), _rays(scale, offset)
    p = _make(scene, scenes.grid_params((0, 0, 0), (10, 10, 10), (2, 2, 2), 64))
    osc = orc.OracleScene(scene)
    want, _ = osc.trace(rays, brute=True)
    assert 0.2 < np.mean(want[:, 1] != 0xFFFFFFFF) < 1.0
    _compare_hits(_gpu_trace(p, rays, 0xFF), want, "closest")
    blocked, _ = osc.trace(rays, any_hit=True, brute=True)
    assert np.array_equal(blocked[:, 1] != 0xFFFFFFFF, _gpu_trace(p, rays, 0xFF, any_hit=True)[:, 1] != 0xFFFFFFFF)
    p.destroy()
