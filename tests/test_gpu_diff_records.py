"""The differentiable gather where its kernels take their other branches: G-buffers whose neighbouring
texels share neither taps nor material, of ragged sizes, against the FP64 oracle; and more texels than
sampling records are kept for, whose weights are recomputed, against a G-buffer small enough for them."""
import numpy as np
import pytest

from oracle import py as orc
from vulkanexp_amd import IrradianceProbes, scenes
from vulkanexp_amd import _lib
from vulkanexp_amd.autograd import DiffContext

pytestmark = pytest.mark.gpu

SKY = scenes.SKY_RADIANCE
M = 96   # material slots; the scene has 65


def _probes():
    scene, grid = scenes.config_small(seed=1, open_top=True)
    p = IrradianceProbes(grid, max_rays_per_probe=128)
    p.set_scene(scene)
    p.set_light(scenes.sun_light())
    p.set_sky(SKY)
    Rs = scenes.orientations(21, 3)
    for R in Rs[:2]:
        p.update(R, _lib.UPDATE_ALL_PROBES)
    p.synchronize()
    return scene, grid, p, Rs[2]


def _texels(scene, n, seed):
    """Points all over the room (a few outside the grid), random normals, views and materials."""
    rng = np.random.Generator(np.random.PCG64(seed))
    unit = lambda: (lambda v: v / np.linalg.norm(v, axis=1, keepdims=True))(rng.normal(size=(n, 3)))
    pos = rng.uniform([-0.5, -0.5, -0.5], [20.5, 10.5, 20.5], (n, 3))
    return [a.astype(np.float32) for a in (pos, unit(), unit())] + [rng.integers(0, len(scene.materials), n).astype(np.int32)]


def _parameters(scene, n, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    albedo = np.zeros((M, 3), np.float32)
    albedo[:len(scene.materials)] = scene.materials["base_color"]
    return albedo, np.array([3.0, 2.5, 2.0], np.float32), rng.uniform(0.0, 0.5, (n, 3)).astype(np.float32)


@pytest.mark.parametrize("n", [1, 63, 65, 1025, 20001])
def test_scattered_texels_match_fp64(n):
    import torch
    scene, grid, p, R = _probes()
    pos, nrm, cam, mat = _texels(scene, n, n)
    albedo, sun, target = _parameters(scene, n, n + 1)
    og, osc = orc.Grid(grid), orc.OracleScene(scene)
    prev, dep, states = p.irradiance()[..., :3].astype(np.float64), p.depth().astype(np.float64), p.states()
    res = osc.update(og, scenes.sun_light(), SKY, R, np.arange(og.count), states, prev.copy(), dep, want_aux=True)
    ref = orc.DiffProblem(og, states, prev, dep, orc.frame_dirs(R, 128), np.arange(og.count), res["aux"].reshape(-1),
                          pos, nrm, cam, mat.astype(np.uint32), M).run(albedo.astype(np.float64), sun.astype(np.float64),
                                                                      target.astype(np.float64), grad=True)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    ctx = DiffContext(p, R, t(pos), t(nrm), t(cam), t(mat), M)
    a, s, tg = t(albedo), t(sun), t(target)
    loss, _ = ctx.forward(a, s, tg)
    ga, gs = ctx.backward(a, s, tg, torch.ones(1, device="cuda"))
    assert abs(float(loss[0]) - ref["loss"]) <= 1e-4 * abs(ref["loss"])
    scale = max(np.abs(ref["g_albedo"]).max(), np.abs(ref["g_sun"]).max())
    assert np.abs(ga.cpu().numpy() - ref["g_albedo"]).max() <= 2e-3 * scale
    assert np.abs(gs.cpu().numpy() - ref["g_sun"]).max() <= 2e-3 * scale
    p.destroy()


def test_more_texels_than_records():
    """700 copies of a 20,736-texel G-buffer (14.5 M texels) have its mean loss and gradients.  A contribution
    is rounded to 2^-50: at most 4.4e-16, alike in every copy; over a copy's 20,736 x 96 contributions that
    sums to 700 x 4.4e-16 / sqrt(3) x sqrt(2.0e6) = 2.5e-10 (rms)."""
    import torch
    scene, _, p, R = _probes()
    n, copies = 20736, 700
    tex = _texels(scene, n, 5)
    albedo, sun, target = _parameters(scene, n, 6)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    state = p.save_state()
    got = []
    for k in (1, copies):
        p.load_state(state)
        pos, nrm, cam = (t(a).repeat(k, 1) for a in tex[:3])
        ctx = DiffContext(p, R, pos, nrm, cam, t(tex[3]).repeat(k), M)
        a, s, tg = t(albedo), t(sun), t(target).repeat(k, 1)
        loss, shade = ctx.forward(a, s, tg)
        ga, gs = ctx.backward(a, s, tg, torch.ones(1, device="cuda"))
        got.append([x.cpu().numpy().astype(np.float64) for x in (loss, ga, gs, shade[:n], shade[-n:])])
    one, many = got
    assert np.array_equal(one[3], many[3]) and np.array_equal(one[3], many[4])
    assert abs(one[0][0] - many[0][0]) <= 1e-5 * one[0][0]
    assert np.abs(one[1] - many[1]).max() <= 5 * 2.5e-10 + 1e-6 * np.abs(one[1]).max()
    assert np.abs(one[2] - many[2]).max() <= 5 * 2.5e-10 + 1e-6 * np.abs(one[2]).max()
    p.destroy()
