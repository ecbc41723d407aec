"""Launches above the four-lane limit (a lane per ray, a wave's last rays handed
to four lanes each) against the oracle or the fp32 format, bit for bit: q8 scenes
of both levels, so that rays are handed on inside an instance and at the top
level, with leaves pending and with stacks that have left the LDS part."""
import numpy as np
import pytest

import lighthouse2_amd as lh
from lighthouse2_amd import scenes
import oracle as orc
from test_gpu_trace import gpu_any, gpu_closest, make_core
from test_gpu_top_level import chain
from test_oracle import _affine, _random_rays, instanced_scene

pytestmark = pytest.mark.gpu
LIMIT = 1 << 17


def spread(rays, seed):
    """The rays several times over in random order, more than a four-lane launch takes (an odd number); which ray each is."""
    pick = np.random.default_rng(seed).integers(0, len(rays), LIMIT + 9001)
    pick[:len(rays)] = np.arange(len(rays))
    return np.ascontiguousarray(rays[pick]), pick


def check(torch, core, rays, closest, occluded, seed=0):
    many, pick = spread(rays, seed)
    assert np.array_equal(gpu_closest(torch, core, many).view(np.uint32), closest.view(np.uint32)[pick])
    assert np.array_equal(gpu_any(torch, core, many), occluded[pick])


def fp32(torch, s, rays):
    core = make_core(s, 0)
    r = gpu_closest(torch, core, rays), gpu_any(torch, core, rays)
    core.Shutdown()
    return r


def test_two_level_against_brute_force(torch_cuda):
    s = instanced_scene(seed=21, meshes=4, instances=40, tris=600)
    o = orc.OracleScene(s)
    rays = _random_rays(np.random.default_rng(2), 30000, -3, 3)
    core = make_core(s, 1)
    check(torch_cuda, core, rays, o.trace(rays, brute=True), o.trace(rays, any_hit=True, brute=True))
    core.Shutdown()


@pytest.mark.parametrize("n", [2, 3, 5, 17, 300])
def test_instance_counts(torch_cuda, n):
    rng = np.random.default_rng(n)
    s = scenes.Scene()
    for k in range(3):
        s.add_mesh(scenes.random_triangles((1, 3, 200)[k], seed=k, sigma=0.2), None)
    for i in range(n):
        s.add_instance(int(rng.integers(3)), _affine(rng))
    rays = _random_rays(rng, 20000, -3, 3)
    o, core = orc.OracleScene(s), make_core(s, 1)
    check(torch_cuda, core, rays, o.trace(rays, brute=True), o.trace(rays, any_hit=True, brute=True), n)
    core.Shutdown()


def test_one_level_against_the_oracle(torch_cuda):
    s = scenes.random_triangle_scene(20000, seed=5)
    o = orc.OracleScene(s)
    rays = _random_rays(np.random.default_rng(7), 40000)
    core = make_core(s, 1)
    check(torch_cuda, core, rays, o.trace(rays), o.trace(rays, any_hit=True))
    core.Shutdown()


@pytest.mark.parametrize("blas,tlas,shrink", [(8, 100, 0), (60, 60, 0), (40, 100, 1), (150, 60, 0)])
def test_deep_trees(torch_cuda, blas, tlas, shrink):
    s = scenes.Scene()
    m = s.add_mesh(chain(blas, 2.0, blas // 2), None)
    for k in range(tlas):
        T = np.eye(4)
        T[:3, :3] *= 2.0 ** -(blas // 2 + 12) if shrink else 1
        T[:3, 3] = np.array([1.0, 0.4, 0.3]) * 1.9 ** (k - tlas // 2)
        s.add_instance(m, T.astype(np.float32).reshape(16))
    rng = np.random.default_rng(blas + tlas)
    rays = np.concatenate([_random_rays(rng, 3000, -f, f) for f in (1, 30, 1e4)])
    aim = np.array([1.0, 0.4, 0.3]) * rng.uniform(0.5, 3, (3000, 1)) * 2.0 ** rng.integers(-20, 20, (3000, 1))
    rays[:3000, 4:7] = (aim - rays[:3000, :3]) / np.linalg.norm(aim - rays[:3000, :3], axis=1, keepdims=True)
    core = make_core(s, 1)
    check(torch_cuda, core, rays, *fp32(torch_cuda, s, rays), seed=blas)
    core.Shutdown()


def shells(n):
    """Nested triangles between a corner's three axes: every box holds the corner."""
    k = np.float32(1.002) ** np.arange(n, dtype=np.float32)
    v = np.ones((n, 3, 4), np.float32)
    v[:, 0, :3], v[:, 1, :3], v[:, 2, :3] = k[:, None] * [1, 0, 0], k[:, None] * [0, 1, 0], k[:, None] * [0, 0, 1]
    return v.reshape(-1, 4)


def deepest_stack(q8, ray):
    """Entries on the stack at most while a ray that hits nothing walks the 4-wide nodes, the nearest child first."""
    f, inv = q8.view(np.float32), 1.0 / ray[4:7].astype(np.float64)
    stack, ref, most = [], 0, 0
    for _ in range(4 * len(q8)):
        if ref & 0x80000000:
            if not stack:
                break
            ref = stack.pop()
            continue
        w = q8[ref]
        step = [f[ref][10], f[ref][11], f[ref][3]]                      # qb.z, qb.w, origin.w
        planes = [(w[4], w[7]), (w[5], w[8]), (w[6], w[9])]             # lo and hi bytes of x, y, z
        hits = []
        for c in range(4):
            if w[12 + c] == 0xffffffff:
                continue
            tn, tf = float(ray[3]), float(ray[7])
            for a in range(3):
                lo, hi = (float(f[ref][a]) + ((int(p) >> (8 * c)) & 255) * float(step[a]) for p in planes[a])
                t = sorted(((lo - ray[a]) * inv[a], (hi - ray[a]) * inv[a]))
                tn, tf = max(tn, t[0]), min(tf, t[1])
            if tn <= tf:
                hits.append((tn, int(w[12 + c])))
        hits.sort(key=lambda h: h[0])
        stack += [r for _, r in hits[:0:-1]]
        most = max(most, len(stack))
        if hits:
            ref = hits[0][1]
        elif stack:
            ref = stack.pop()
        else:
            break
    return most


@pytest.mark.parametrize("two_level", [False, True])
def test_stacks_beyond_the_lds_part(torch_cuda, two_level):
    """Stacks leave the 16 entries in LDS (shown by walking the nodes), so a wave's last rays are handed on with spilled entries."""
    s = scenes.Scene()
    m = s.add_mesh(shells(4096), None)
    if two_level:
        rng = np.random.default_rng(3)
        for k in range(12):
            T = np.eye(4)
            T[:3, :3] *= rng.uniform(0.9, 1.1)
            T[:3, 3] = rng.uniform(-1, 1, 3)
            s.add_instance(m, T.astype(np.float32).reshape(16))
    else:
        s.add_instance(m)
    rng = np.random.default_rng(1)
    n = 3000
    d = np.abs(rng.standard_normal((n, 3))).astype(np.float32) + np.float32(0.2)
    rays = np.zeros((n, 8), np.float32)
    rays[:, 4:7], rays[:, 7] = d / np.linalg.norm(d, axis=1, keepdims=True), 1e30
    rays[: n // 3, 7] = 0.5                                  # end before the first shell: every box holds the origin, nothing is hit
    rays[n // 3: 2 * n // 3, 3] = rng.uniform(0.6, 2000, len(rays[n // 3: 2 * n // 3]))   # start between two shells
    core = make_core(s, 1)
    q8 = core.bvh_layout_download(0)[1]
    assert min(deepest_stack(q8, r.astype(np.float64)) for r in rays[: n // 3: n // 12]) > 16
    closest, occluded = fp32(torch_cuda, s, rays)
    assert len(np.unique(closest.view(np.int32)[:, 2])) > 500
    check(torch_cuda, core, rays, closest, occluded)
    core.Shutdown()
