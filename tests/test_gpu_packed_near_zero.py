"""Rays whose direction has components at or near zero: closest hits equal the oracle's brute-force scan bit
for bit, down to components whose reciprocals overflow, and a sun straight overhead costs the shadow rays as
many node visits as one a thousandth of a radian beside it (the same rays to 0.03 of a scene unit, so within
5 %)."""
import numpy as np
import pytest

from oracle import py as orc
from vulkanexp_amd import scenes
from vulkanexp_amd import _lib

pytestmark = pytest.mark.gpu


def _rays(n, small, seed):
    """Rays along a coordinate axis; the other components of magnitude `small`, of either sign."""
    rng = np.random.Generator(np.random.PCG64(seed))
    d = np.where(rng.random((n, 3)) < 0.5, -small, small).astype(np.float32)
    d[np.arange(n), rng.integers(0, 3, n)] = np.where(rng.random(n) < 0.5, -1.0, 1.0)
    r = np.zeros((n, 8), np.float32)
    r[:, :3], r[:, 4:7], r[:, 7] = rng.uniform([0.2, 0.2, 0.2], [19.8, 9.8, 19.8], (n, 3)), d, 1e5
    return r


@pytest.mark.parametrize("small", [0.0, 1e-44, 1e-38, 1e-37, 1e-36, 1e-30, 1e-20, 1e-7])
def test_hits_with_components_near_zero(small):
    from test_gpu_parity import _compare_hits, _gpu_trace, _make
    scene, grid = scenes.config_small(seed=1)
    rays = _rays(4000, np.float32(small), 31)
    p, osc = _make(scene, grid), orc.OracleScene(scene)
    want, _ = osc.trace(rays, brute=True)
    assert np.mean(want[:, 1] != 0xFFFFFFFF) > 0.9
    _compare_hits(_gpu_trace(p, rays, 0xFF), want, "closest")
    blocked, _ = osc.trace(rays, any_hit=True, brute=True)
    assert np.array_equal(blocked[:, 1] != 0xFFFFFFFF, _gpu_trace(p, rays, 0xFF, any_hit=True)[:, 1] != 0xFFFFFFFF)
    p.destroy()


def test_overhead_sun_visits_no_more_nodes():
    from test_gpu_parity import _make
    scene = scenes.clustered_scene(seed=5, n_instances=24)
    p = _make(scene, scenes.grid_params(*scenes.inset_extent(scene), (8, 4, 8), 64))
    R = scenes.orientations(3, 1)[0]
    visits = []
    for travel in ((1e-3, -1.0, 1e-3), (0.0, -1.0, 0.0), (0.0, -1.0, 1e-38)):
        p.set_light(scenes.sun_light(travel))
        p.update(R, _lib.UPDATE_ALL_PROBES | _lib.UPDATE_COUNT_VISITS)
        p.synchronize()
        st = p.trace_stats()
        visits.append(st["shadow_nodes"] / st["shadow_rays"])
    print(visits)
    assert visits[0] > 1.0
    assert abs(visits[1] - visits[0]) <= 0.05 * visits[0] and abs(visits[2] - visits[0]) <= 0.05 * visits[0]
    p.destroy()
