"""Gradient sums are exact: contributions of either sign far above 8.0 (where doubles no longer hold every
multiple of 2^-50) that cancel leave the gradients of the others unchanged, bit for bit, and so does the order
of the texels."""
import numpy as np
import pytest

from test_gpu_diff_records import M, _parameters, _probes, _texels
from vulkanexp_amd.autograd import DiffContext

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,alike", [(64, False), (6912, False), (1000, True)])
def test_large_contributions_cancel_exactly(n, alike):
    """alike: texels of one probe cell with one normal and material, whose contributions share their sums."""
    import torch
    scene, _, p, R = _probes()
    tex = _texels(scene, n, 11)
    if alike:
        tex[0][:] = tex[0] * 0.05 + np.float32([9.0, 5.0, 9.0])
        tex[1][:], tex[3][:] = tex[1][0], tex[3][0]
    albedo, sun, target = _parameters(scene, n, 12)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    a, s, one = t(albedo), t(sun), torch.ones(1, device="cuda")
    pos, nrm, cam, mat = (t(x).repeat(3, *[1] * (x.ndim - 1)) for x in tex)
    state = p.save_state()

    def context(order):
        p.load_state(state)
        return DiffContext(p, R, pos[order].contiguous(), nrm[order].contiguous(), cam[order].contiguous(),
                           mat[order].contiguous(), M)

    ident = torch.arange(3 * n, device="cuda")
    ctx = context(ident)
    _, shade = ctx.forward(a, s, t(target).repeat(3, 1))
    shade = shade[:n]
    big = torch.full_like(shade, float(2 ** 26))
    assert torch.equal(shade - big, -big) and torch.equal(shade + big, big)  # the errors are +-big exactly
    quiet, loud = torch.cat([shade, shade, t(target)]), torch.cat([big, -big, t(target)])
    want = ctx.backward(a, s, quiet.contiguous(), one)
    assert float(want[0].abs().max()) > 0.0
    got = ctx.backward(a, s, loud.contiguous(), one)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    order = torch.from_numpy(np.random.Generator(np.random.PCG64(13)).permutation(3 * n)).cuda()
    ctx = context(order)
    ctx.forward(a, s, loud[order].contiguous())
    got = ctx.backward(a, s, loud[order].contiguous(), one)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    p.destroy()
