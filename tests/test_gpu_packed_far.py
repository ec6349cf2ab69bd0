"""Rays from far away past small details, whose nodes have fewer than four children: closest hits equal the
oracle's brute-force scan bit for bit, and any-hit decisions agree."""
import numpy as np
import pytest

from oracle import py as orc
from vulkanexp_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size,reach", [(1e-4, 1e5), (1e-6, 1e4), (1e-3, 1e6), (1e-5, 1e9)])
def test_hits_past_small_details(size, reach):
    from test_gpu_parity import _compare_hits, _gpu_trace, _make
    from test_packed_host import _details
    scene, n = _details(size), 4000
    rng = np.random.Generator(np.random.PCG64(9))
    to = np.stack([rng.uniform(0, 64 * size, n), rng.uniform(2 * size, 3 * size, n), rng.uniform(0, 40 * size, n)], 1)
    to += 1e-7 * reach * rng.uniform(-1.0, 1.0, (n, 3))
    up = rng.normal(size=(n, 3))
    up /= np.linalg.norm(up, axis=1, keepdims=True)
    up[:, 1] = np.abs(up[:, 1]) + 0.1
    rays = np.zeros((n, 8), np.float32)
    rays[:, :3] = to + reach * up
    rays[:, 4:7] = (to - rays[:, :3].astype(np.float64)) / reach
    rays[:, 7] = 1e3 * reach
    p = _make(scene, scenes.grid_params((-90, 0, -90), (90, 1, 90), (2, 2, 2), 64))
    osc = orc.OracleScene(scene)
    want, _ = osc.trace(rays, brute=True)
    assert np.mean(want[:, 1] != 0xFFFFFFFF) > 0.3
    _compare_hits(_gpu_trace(p, rays, 0xFF), want, "closest")
    blocked, _ = osc.trace(rays, any_hit=True, brute=True)
    assert np.array_equal(blocked[:, 1] != 0xFFFFFFFF, _gpu_trace(p, rays, 0xFF, any_hit=True)[:, 1] != 0xFFFFFFFF)
    p.destroy()
