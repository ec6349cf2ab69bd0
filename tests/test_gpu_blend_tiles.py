"""The blend's workgroup shapes agree bit for bit.

launch_blend picks 16-probe tiles (k_blend_tile), 4-wave FP32 blocks (k_blend_fp32) or 64-probe workgroups
(k_blend_wide) by the number of listed probes.  Each issues the same MFMAs per output element in the same
order on equally rounded operands, so the tiles of a probe must not depend on how many others are listed.
"""
import numpy as np
import pytest

import vulkanexp_amd as ddgi
from vulkanexp_amd import _lib, scenes

pytestmark = pytest.mark.gpu

FLAGS = {"fp32": 0, "bf16": _lib.UPDATE_BLEND_BF16, "fp16": _lib.UPDATE_BLEND_FP16}


@pytest.mark.parametrize("mode", list(FLAGS))
@pytest.mark.parametrize("rays", [33, 100, 512])
def test_listed_count_does_not_change_a_tile(mode, rays):
    """A volume of 80 probes per compute unit: whole (tiles, three rounds), then its first 1 and 17 probes
    and 32 per unit (tiles), 32 per unit + 1 and 48 per unit (FP32: blocks) and 64 per unit (wide), listed in a
    shuffled order; ray records with misses, back faces and out-of-range distances; a last K step that is
    partial (33, 100) and one that is full (512)."""
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    res = (32, 80 * cus // 1024, 32)
    lo, hi = np.zeros(3), np.ones(3)
    p = ddgi.IrradianceProbes(np.array(scenes.grid_params(lo, hi, res, rays)), max_rays_per_probe=rays)
    P = p.get_probe_count()
    assert P >= 79 * cus
    rng = np.random.Generator(np.random.PCG64(rays))
    buf = rng.random((P, rays, 4), dtype=np.float32)
    buf[..., 3] = rng.random((P, rays), dtype=np.float32) * 0.2 - 0.02  # cells are about 0.05 wide
    idx = rng.permutation(P).astype(np.uint32)
    R = scenes.orientations(90 + rays, 1)[0]
    rays_d, idx_d = torch.from_numpy(buf).cuda(), torch.from_numpy(idx.view(np.int32)).cuda()
    p.blend_rays(rays_d, idx_d, R, FLAGS[mode])  # exposed tiles that are not zero
    state = p.save_state()
    whole = None
    for count in (P, 1, 17, 32 * cus, 32 * cus + 1, 48 * cus, 64 * cus):
        p.load_state(state)
        p.blend_rays(rays_d[:count].contiguous(), idx_d[:count].contiguous(), R, FLAGS[mode])
        p.synchronize()
        sel = idx[:count].astype(np.int64)
        out = [p.irradiance(_lib.LAYOUT_TILED), p.depth(_lib.LAYOUT_TILED), p.states()]
        if whole is None:
            whole = out
            assert np.isfinite(whole[0]).all() and whole[0][..., :3].max() > 0
        for a, b, what in zip(out, whole, ("irradiance", "depth", "states")):
            assert np.array_equal(a[sel], b[sel]), f"{mode}, {rays} rays, {count} listed: {what}"
    p.destroy()
