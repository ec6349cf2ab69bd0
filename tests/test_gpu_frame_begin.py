"""The start of an update: ray directions, thread order, blend weights and probe list from one launch,
at the ray counts where the ranking splits its comparisons differently (128, 256 and their neighbours)
and where the weight rows are padded."""
import numpy as np
import pytest

from vulkanexp_amd import IrradianceProbes, _lib, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rays", [1, 2, 63, 65, 128, 129, 256, 257, 511, 512])
def test_order_list_and_weights(rays):
    """A partial update and then a whole one (the list is rebuilt) of a 5 x 3 x 4 volume.  The order sorts the
    stored directions by elevation, ties by index, and the lists are what they should be.  Blending the same
    records in ray-index order gives the same tiles up to the order of the FP32 sums of up to 512 positive
    terms: 2e-5 of the largest value, the bound of the FP32 blend against FP64 (twice, one per side)."""
    import torch
    scene, _ = scenes.config_small(seed=9, rays=64, open_top=True)
    lo, hi = scenes.inset_extent(scene)
    p = IrradianceProbes(np.array(scenes.grid_params(lo, hi, (5, 3, 4), rays)), max_rays_per_probe=rays, probes_per_update=7)
    p.set_scene(scene)
    p.set_light(scenes.sun_light())
    p.set_sky(scenes.SKY_RADIANCE)
    R = scenes.orientations(rays, 3)
    p.update(R[0], _lib.UPDATE_ALL_PROBES)
    p.update(R[1], 0)
    p.synchronize()
    _, idx = p.last_update_rays()
    assert 0 < len(idx) <= 7 and len(set(idx.tolist())) == len(idx)
    state = p.save_state()
    p.update(R[2], _lib.UPDATE_ALL_PROBES)
    p.synchronize()
    rec, idx = p.last_update_rays()
    assert np.array_equal(idx, np.arange(60, dtype=np.uint32))
    view = p.device_view()
    from vulkanexp_amd.probes import _device_copy
    dirs = _device_copy(view.ray_directions, rays * 4, torch.float32).numpy().reshape(rays, 4)
    assert np.array_equal(p._ray_order(view, rays), np.argsort(dirs[:, 1], kind="stable"))
    assert np.allclose(np.linalg.norm(dirs[:, :3], axis=1), 1.0, atol=1e-5)
    got = [p.irradiance(_lib.LAYOUT_TILED), p.depth(_lib.LAYOUT_TILED)]
    p.load_state(state)
    p.blend_rays(torch.from_numpy(rec).cuda(), torch.from_numpy(idx.view(np.int32)).cuda(), R[2], _lib.UPDATE_ALL_PROBES)
    p.synchronize()
    for a, b in zip(got, [p.irradiance(_lib.LAYOUT_TILED), p.depth(_lib.LAYOUT_TILED)]):
        assert np.abs(a - b).max() <= 4e-5 * max(np.abs(a).max(), 1e-6)
    p.destroy()
