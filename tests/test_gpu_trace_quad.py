"""The four-lanes-per-ray traversal of small launches against the oracle (bit
for bit): ray counts at the edges of its waves and of the rule that picks it,
leaves of more than four triangles, ties, and stacks beyond the LDS part."""
import numpy as np
import pytest

import lighthouse2_amd as lh
from lighthouse2_amd import scenes
import oracle as orc
from test_oracle import _random_rays, instanced_scene
from test_gpu_trace import gpu_any, gpu_closest, make_core

pytestmark = pytest.mark.gpu
LIMIT = 1 << 17          # largest launch that takes four lanes per ray


def check(torch, core, o, rays):
    got = gpu_closest(torch, core, rays)
    assert np.array_equal(got.view(np.uint32), o.trace(rays).view(np.uint32)), len(rays)
    assert np.array_equal(gpu_any(torch, core, rays), o.trace(rays, any_hit=True)), len(rays)


@pytest.mark.parametrize("two_level", [False, True])
def test_ray_counts(torch_cuda, two_level):
    s = instanced_scene(seed=4, meshes=3, instances=25, tris=500) if two_level else scenes.random_triangle_scene(4000, seed=9)
    o, core = orc.OracleScene(s), make_core(s, 1)
    rays = _random_rays(np.random.default_rng(2), 20000)
    for n in (1, 2, 3, 16, 17, 31, 33, 1023, 1024, 1025, 2048, 4097, 16385, 20000):
        check(torch_cuda, core, o, rays[:n])
    core.Shutdown()


@pytest.mark.parametrize("n", [LIMIT - 1, LIMIT, LIMIT + 1])
def test_both_sides_of_the_rule_agree(torch_cuda, n):
    """The largest four-lane launch and the smallest of the other kind: the same records for the same rays."""
    s = scenes.random_triangle_scene(3000, seed=11)
    core = make_core(s, 1)
    rays = _random_rays(np.random.default_rng(5), LIMIT + 1)
    few = gpu_closest(torch_cuda, core, rays[:n])
    parts = np.concatenate([gpu_closest(torch_cuda, core, rays[:70000]), gpu_closest(torch_cuda, core, rays[70000:n])])
    assert np.array_equal(few.view(np.uint32), parts.view(np.uint32))
    m = gpu_any(torch_cuda, core, rays[:n])
    assert np.array_equal(m, few.view(np.int32)[:, 2] >= 0)
    core.Shutdown()


@pytest.mark.parametrize("copies", [3, 4, 5, 9, 255])
def test_leaves_of_coincident_triangles(torch_cuda, copies):
    """Identical triangles share a centroid and one leaf (up to 255): every hit is a tie, the smallest primitive id wins."""
    base = np.array([[0, 0, 0, 1], [1, 0, 0, 1], [0, 1, 0, 1]], np.float32)
    far = base + np.float32([0, 0, 5, 0])
    s = scenes.Scene()
    s.add_instance(s.add_mesh(np.concatenate([far] + [base] * copies), None))
    o, core = orc.OracleScene(s), make_core(s, 1)
    rng = np.random.default_rng(copies)
    rays = np.zeros((200, 8), np.float32)
    rays[:, :2] = rng.uniform(-0.1, 1.1, (200, 2))
    rays[:, 2], rays[:, 6], rays[:, 7] = -1.0, 1.0, 1e30
    rays[100:, 3] = 2.0                                     # starts beyond the pile: only the far triangle counts
    check(torch_cuda, core, o, rays)
    got = gpu_closest(torch_cuda, core, rays).view(np.int32)[:, 2]
    assert set(got[:100]) <= {-1, 1} and 1 in got[:100] and set(got[100:]) <= {-1, 0}
    core.Shutdown()


def test_deep_stack(torch_cuda):
    """Nested shells seen from their common corner: every node's children overlap, so stacks grow past the LDS part."""
    n = 4096
    k = np.float32(1.002) ** np.arange(n, dtype=np.float32)
    v = np.ones((n, 3, 4), np.float32)
    v[:, 0, :3], v[:, 1, :3], v[:, 2, :3] = k[:, None] * [1, 0, 0], k[:, None] * [0, 1, 0], k[:, None] * [0, 0, 1]
    s = scenes.Scene()
    s.add_instance(s.add_mesh(v.reshape(-1, 4), None))
    o, core = orc.OracleScene(s), make_core(s, 1)
    rng = np.random.default_rng(1)
    d = np.abs(rng.standard_normal((500, 3))).astype(np.float32)
    rays = np.zeros((500, 8), np.float32)
    rays[:, :3] = d * 5000
    rays[:, 4:7] = -d / np.linalg.norm(d, axis=1, keepdims=True)
    rays[:, 7] = 1e30
    rays[250:, :3], rays[250:, 4:7] = 0.0, -rays[250:, 4:7]
    check(torch_cuda, core, o, rays)
    core.Shutdown()
