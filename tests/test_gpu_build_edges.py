"""The BVH builder at the edges of its two kinds of nodes (512 primitives per
wave, 2,048 per chunk of a larger node) and with coincident centroids, whose
ranges are halved by position: the tree equals the oracle's, and hits through
the top level equal the oracle's."""
import numpy as np
import pytest

import lighthouse2_amd as lh
from lighthouse2_amd import scenes
import oracle as orc
from test_gpu_trace import canonical, gpu_closest, make_core
from test_oracle import _random_rays

pytestmark = pytest.mark.gpu


def check_tree(scene):
    core = make_core(scene, 1)
    gn, gp = core.bvh_download(0)
    on, op, _ = orc.OracleScene(scene).bvh_nodes(0)
    assert len(gn) == len(on) and canonical(gn, gp) == canonical(on, op)
    return core


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 63, 64, 65, 128, 511, 512, 513, 1025, 2047, 2048, 2049, 4097, 9000])
def test_tree_equals_oracle(torch_cuda, n):
    check_tree(scenes.random_triangle_scene(n, seed=n)).Shutdown()


def test_a_mesh_rebuilt_smaller_and_larger(torch_cuda):
    """One core's workspace and node arrays reused by other sizes."""
    core = lh.RenderCore()
    core.SetMaterials(lh.formats.lambert_material((0.5, 0.5, 0.5)))
    for n in (3000, 40, 9000, 700, 3000):
        s = scenes.random_triangle_scene(n, seed=n + 1)
        core.SetGeometry(0, s.meshes[0][0])
        core.SetInstance(0, 0)
        core.FinalizeInstances()
        gn, gp = core.bvh_download(0)
        o = orc.OracleScene(s)
        on, op, _ = o.bvh_nodes(0)
        assert canonical(gn, gp) == canonical(on, op)
        rays = _random_rays(np.random.default_rng(n), 500)
        assert np.array_equal(gpu_closest(torch_cuda, core, rays).view(np.uint32), o.trace(rays).view(np.uint32))
    core.Shutdown()


@pytest.mark.parametrize("n", [256, 512, 513, 1500, 5000])
def test_coincident_triangles_are_halved(torch_cuda, n):
    base = np.array([[0, 0, 0, 1], [1, 0, 0, 1], [0, 1, 0, 1]], np.float32)
    s = scenes.Scene()
    s.add_instance(s.add_mesh(np.concatenate([base] * n), None))
    check_tree(s).Shutdown()


def test_clustered_and_flat_geometry(torch_cuda):
    """All centroids in a plane (one invalid axis), half of them in one point."""
    rng = np.random.default_rng(5)
    c = np.zeros((1400, 1, 3), np.float32)
    c[:700, 0, :2] = rng.random((700, 2))
    v = np.ones((1400, 3, 4), np.float32)
    v[:, :, :3] = c + np.float32([[[0, 0, 0], [0.01, 0, 0], [0, 0.01, 0]]])
    s = scenes.Scene()
    s.add_instance(s.add_mesh(v.reshape(-1, 4), None))
    core, o = make_core(s, 1), orc.OracleScene(s)
    rays = np.zeros((300, 8), np.float32)
    rays[:, :2], rays[:, 2], rays[:, 6], rays[:, 7] = rng.random((300, 2)), -1.0, 1.0, 10.0
    rays[:50, :2] = 0.002
    assert np.array_equal(gpu_closest(torch_cuda, core, rays).view(np.uint32), o.trace(rays).view(np.uint32))
    core.Shutdown()


@pytest.mark.parametrize("instances", [2, 65, 600, 1300])
def test_top_level_of_coincident_and_spread_instances(torch_cuda, instances):
    """One instance per leaf: coincident instances are split down to one."""
    v = scenes.random_triangles(50, seed=3, sigma=0.2)
    s = scenes.Scene()
    m = s.add_mesh(v, None)
    rng = np.random.default_rng(instances)
    for k in range(instances):
        T = np.eye(4, dtype=np.float32)
        if k % 2:
            T[:3, 3] = rng.uniform(-5, 5, 3)
        s.add_instance(m, T.reshape(16))
    core, o = make_core(s, 1), orc.OracleScene(s)
    rays = _random_rays(rng, 3000, -6, 6)
    assert np.array_equal(gpu_closest(torch_cuda, core, rays).view(np.uint32), o.trace(rays).view(np.uint32))
    core.Shutdown()
