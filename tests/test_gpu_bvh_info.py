"""The BVH's reported size is that of the arrays the traversal reads."""
import pytest

from vulkanexp_amd import IrradianceProbes, scenes
from vulkanexp_amd import _lib

pytestmark = pytest.mark.gpu


def test_bytes_are_those_of_nodes_and_slots():
    scene, grid = scenes.config_small(seed=1)
    p = IrradianceProbes(grid, max_rays_per_probe=128)
    p.set_scene(scene)
    info = p.bvh_info()
    assert info["nodes"] > 0 and info["triangles"] >= scene.triangle_count
    assert info["bytes"] == info["nodes"] * _lib.NODE_BYTES + info["triangles"] * _lib.TRIANGLE_BYTES
    p.destroy()
