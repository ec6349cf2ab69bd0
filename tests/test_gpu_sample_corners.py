"""sampleProbes at few points (eight lanes per point) and at many (one thread per point): the same bits."""
import numpy as np
import pytest

from vulkanexp_amd import IrradianceProbes, _lib, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 7, 8, 33, 4097, 65536])
def test_both_kernels_give_the_same_samples(count):
    """65537 points (one thread each), some outside the grid, on its boundary or not finite, then their first
    `count` (eight lanes each); a third of the probes off, so that corners drop out."""
    import torch
    scene, _ = scenes.config_small(seed=13, rays=64, open_top=True)
    lo, hi = scenes.inset_extent(scene)
    p = IrradianceProbes(np.array(scenes.grid_params(lo, hi, (7, 4, 6), 64)), max_rays_per_probe=64)
    p.set_scene(scene)
    p.set_light(scenes.sun_light())
    p.set_sky(scenes.SKY_RADIANCE)
    for R in scenes.orientations(14, 2):
        p.update(R, _lib.UPDATE_ALL_PROBES)
    p.synchronize()
    rng = np.random.Generator(np.random.PCG64(15))
    states = p.states().copy()
    states[rng.random(len(states)) < 0.33] = 0
    p.set_states(states)
    lo, hi = np.asarray(lo, np.float32), np.asarray(hi, np.float32)
    pos = lo + (rng.random((65537, 3)) * 1.2 - 0.1).astype(np.float32) * (hi - lo)
    pos[1], pos[2], pos[3, 0], pos[4, 1], pos[5, 2], pos[6, 0] = lo, hi, np.nan, np.inf, 1e30, 4e9
    n, v = (w / np.linalg.norm(w, axis=1, keepdims=True) for w in rng.normal(size=(2, 65537, 3)))
    args = [torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda() for a in (pos, n, v)]
    many = p.sample(*args).cpu().numpy()
    few = p.sample(*[a[:count].contiguous() for a in args]).cpu().numpy()
    assert np.array_equal(few, many[:count], equal_nan=True)
    assert (many[4:7] == 0).all()  # beyond the grid, however far: no probe contributes
    assert (many > 0).any()
    p.destroy()
