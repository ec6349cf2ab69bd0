"""A prepared differentiable context keeps its frame: updates of the same probes with other orientations, and
another number of rays, between its calls change neither loss nor gradients."""
import numpy as np
import pytest

from test_gpu_diff_records import M, _parameters, _probes, _texels
from vulkanexp_amd import scenes
from vulkanexp_amd import _lib
from vulkanexp_amd.autograd import DiffContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rays", [128, 96])
def test_updates_between_the_calls_change_nothing(rays):
    import torch
    scene, _, p, R = _probes()
    n = 2000
    pos, nrm, cam, mat = _texels(scene, n, 3)
    albedo, sun, target = _parameters(scene, n, 4)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    ctx = DiffContext(p, R, t(pos), t(nrm), t(cam), t(mat), M)
    a, s, tg, one = t(albedo), t(sun), t(target), torch.ones(1, device="cuda")
    want = [x.cpu() for x in (*ctx.forward(a, s, tg), *ctx.backward(a, s, tg, one))]
    p.GridParameters["rays_per_probe"] = rays
    p.update_uniforms()
    for other in scenes.orientations(77, 3):
        p.update(other, _lib.UPDATE_ALL_PROBES)
        got = [x.cpu() for x in (*ctx.forward(a, s, tg), *ctx.backward(a, s, tg, one))]
        assert all(torch.equal(x, y) for x, y in zip(want, got))
    p.destroy()
