"""Tiles of the probes that a partial update leaves out: the next atlases start as copies of the exposed ones,
made by extra workgroups of the shading launch."""
import numpy as np
import pytest

from vulkanexp_amd import IrradianceProbes, _lib, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res", [(2, 2, 2), (5, 3, 7), (16, 9, 15)])  # far below, above and off a copy workgroup's 1024
@pytest.mark.parametrize("flags", [0, _lib.UPDATE_HYSTERESIS_RAMP, _lib.UPDATE_NO_TIMING | _lib.UPDATE_HYSTERESIS_RAMP])
def test_unlisted_tiles_stay(res, flags):
    """Three partial updates in a row (each publishes the other buffer): bytes of unlisted tiles and states
    unchanged, at least one listed tile new."""
    scene, _ = scenes.config_small(seed=11, rays=64, open_top=True)
    lo, hi = scenes.inset_extent(scene)
    p = IrradianceProbes(np.array(scenes.grid_params(lo, hi, res, 64)), max_rays_per_probe=64,
                         probes_per_update=max(1, int(np.prod(res)) // 3))
    p.set_scene(scene)
    p.set_light(scenes.sun_light())
    p.set_sky(scenes.SKY_RADIANCE)
    R = scenes.orientations(12, 5)
    p.update(R[0], _lib.UPDATE_ALL_PROBES)

    def read():
        p.synchronize()
        return [p.irradiance(_lib.LAYOUT_TILED).copy(), p.depth(_lib.LAYOUT_TILED).copy(), p.states().copy()]

    listed = 0
    before = read()
    for r in R[1:4]:
        p.update(r, flags)
        now = read()
        view = p.device_view()
        import torch
        from vulkanexp_amd.probes import _device_copy
        all_idx = _device_copy(view.probe_indices, p.get_probe_count(), torch.int32).numpy().view(np.uint32)
        changed = (now[0] != before[0]).reshape(len(now[0]), -1).any(1) | (now[1] != before[1]).reshape(len(now[1]), -1).any(1)
        bound = max(1, p.get_probe_count() // 3)
        assert set(np.flatnonzero(changed)) <= set(all_idx[:bound].tolist())
        assert set(np.flatnonzero(now[2] != before[2])) <= set(all_idx[:bound].tolist())
        listed += int(changed.sum())
        before = now
    assert listed > 0
    p.destroy()


def test_ramped_partial_update_is_refused_under_capture():
    """It reads the number of updated probes back, so it cannot be captured: an error, nothing enqueued."""
    import torch
    scene, _ = scenes.config_small(seed=11, rays=64)
    lo, hi = scenes.inset_extent(scene)
    p = IrradianceProbes(np.array(scenes.grid_params(lo, hi, (4, 3, 4), 64)), max_rays_per_probe=64, probes_per_update=9)
    p.set_scene(scene)
    p.set_light(scenes.sun_light())
    R = scenes.orientations(12, 1)[0]
    p.update(R, _lib.UPDATE_ALL_PROBES)
    p.update(R, _lib.UPDATE_HYSTERESIS_RAMP)
    p.synchronize()
    graph, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    x = torch.zeros(4, device="cuda")
    with torch.cuda.graph(graph, stream=s):
        x.add_(1.0)
        with pytest.raises(Exception, match="captured"):
            p.update(R, _lib.UPDATE_HYSTERESIS_RAMP | _lib.UPDATE_NO_TIMING, stream=s)
    graph.replay()
    torch.cuda.synchronize()
    assert x[0].item() == 1.0
    p.update(R, _lib.UPDATE_HYSTERESIS_RAMP)
    p.synchronize()
    p.destroy()
