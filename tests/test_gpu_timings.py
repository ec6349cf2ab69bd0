"""Phase timings come from stamps the kernels store: plausible for every launch shape that stores them."""
import time

import numpy as np
import pytest

from vulkanexp_amd import IrradianceProbes, _lib, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, _lib.UPDATE_BLEND_BF16, _lib.UPDATE_BLEND_FP16])
@pytest.mark.parametrize("res,rays", [((3, 2, 3), 64), ((16, 9, 16), 320), ((32, 12, 32), 64)])  # tiles; ordered; blocks and wide
def test_phases_add_up(res, rays, mode):
    """Phases are not negative and add up to the total (each is a float of whole 10 ns ticks), the traced and
    blended ones are positive, and the total lies within the host's time around it; an update without timings
    in between leaves the last ones; a blend alone has only its own phase."""
    import torch
    scene, _ = scenes.config_small(seed=17, rays=64, open_top=True)
    lo, hi = scenes.inset_extent(scene)
    p = IrradianceProbes(np.array(scenes.grid_params(lo, hi, res, rays)), max_rays_per_probe=rays,
                         probes_per_update=max(1, int(np.prod(res)) // 2))
    p.set_scene(scene)
    p.set_light(scenes.sun_light())
    R = scenes.orientations(18, 1)[0]
    p.update(R, _lib.UPDATE_ALL_PROBES | mode)
    p.synchronize()
    for flags in (_lib.UPDATE_ALL_PROBES, 0, _lib.UPDATE_HYSTERESIS_RAMP):
        t0 = time.perf_counter()
        p.update(R, flags | mode)
        t = p.timings()
        wall = (time.perf_counter() - t0) * 1e3
        parts = [t[k] for k in ("select_ms", "primary_ms", "shade_ms", "blend_ms")]
        assert min(parts) >= 0 and min(parts[1:]) > 0
        assert abs(sum(parts) - t["total_ms"]) <= 1e-5 * t["total_ms"] + 1e-6
        assert t["total_ms"] < wall
    p.update(R, mode)
    p.update(R, mode | _lib.UPDATE_NO_TIMING)
    a = p.timings()
    p.update(R, mode | _lib.UPDATE_NO_TIMING)
    p.synchronize()
    assert p.timings() == a
    P = p.get_probe_count()
    buf = torch.rand((P, rays, 4), device="cuda")
    idx = torch.arange(P, dtype=torch.int32, device="cuda")
    p.blend_rays(buf, idx, R, mode)
    t = p.timings()
    assert t["blend_ms"] == t["total_ms"] > 0 and t["primary_ms"] == t["select_ms"] == 0
    p.destroy()
