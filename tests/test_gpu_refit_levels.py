"""Instance moves on trees whose box hierarchy has one, two and three launches' worth of levels (512 slots
per three): after the moves, and after moving back, the hits equal those of a handle built from the same
transforms, bit for bit."""
import dataclasses

import numpy as np
import pytest

from vulkanexp_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("instances", [1, 3, 40, 300])
def test_moved_instances_trace_like_a_rebuilt_scene(instances):
    from test_gpu_parity import _gpu_trace, _make
    scene = scenes.clustered_scene(7, n_instances=instances)
    rng = np.random.Generator(np.random.PCG64(instances))
    M = scene.instances["transform"].reshape(-1, 3, 4).astype(np.float64)
    a = rng.uniform(-1.0, 1.0, len(M))
    rot = np.zeros((len(M), 3, 3))
    rot[:, 0, 0] = rot[:, 2, 2] = np.cos(a)
    rot[:, 0, 2], rot[:, 2, 0], rot[:, 1, 1] = np.sin(a), -np.sin(a), 1.0
    new = M.copy()
    new[:, :, :3] = rot @ M[:, :, :3]
    new[:, :, 3] += rng.uniform(-1.0, 1.0, (len(M), 3))
    new = new.astype(np.float32).reshape(-1, 12)
    inst = scene.instances.copy()
    inst["transform"] = new
    n = 20000
    rays = np.zeros((n, 8), np.float32)
    rays[:, :3] = rng.uniform([-2, -2, -2], [62, 20, 42], (n, 3))
    d = rng.normal(size=(n, 3))
    rays[:, 4:7], rays[:, 7] = d / np.linalg.norm(d, axis=1, keepdims=True), 200.0
    grid = scenes.grid_params((0, 0, 0), (10, 10, 10), (2, 2, 2), 64)
    p, q = _make(scene, grid), _make(dataclasses.replace(scene, instances=inst), grid)
    before = _gpu_trace(p, rays, 0xFF)
    p.update_instances(0, new)
    assert np.array_equal(_gpu_trace(p, rays, 0xFF), _gpu_trace(q, rays, 0xFF))
    half = len(M) // 2
    p.update_instances(0, scene.instances["transform"][:half])
    p.update_instances(half, scene.instances["transform"][half:])
    assert np.array_equal(_gpu_trace(p, rays, 0xFF), before)
    assert 0.05 < np.mean(before[:, 1] != 0xFFFFFFFF)
    p.destroy()
    q.destroy()
