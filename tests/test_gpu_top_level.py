"""The 4-wide top level: every arity of its nodes, instances that need the exact
boxes (the whole scene then runs on fp32 nodes) and trees too deep for a wide
node per binary level. Hits equal the fp32 format's and the oracle's brute
force bit for bit, in launches of a quad and of a lane per ray."""
import numpy as np
import pytest

import lighthouse2_amd as lh
from lighthouse2_amd import scenes
import oracle as orc
from test_gpu_trace import gpu_any, gpu_closest, make_core
from test_oracle import _affine, _random_rays

pytestmark = pytest.mark.gpu


def both(torch, s, rays, loops=(0, 1, 2)):
    """q8 hits of every loop; equal to the fp32 format's."""
    core = make_core(s, 0)
    want, bits = gpu_closest(torch, core, rays), gpu_any(torch, core, rays)
    core.Shutdown()
    for loop in loops:
        core = make_core(s, 1, loop)
        assert np.array_equal(gpu_closest(torch, core, rays).view(np.uint32), want.view(np.uint32)), loop
        assert np.array_equal(gpu_any(torch, core, rays), bits), loop
        core.Shutdown()
    return want


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6, 7, 17, 64, 65, 300])
def test_instance_counts(torch_cuda, n):
    rng = np.random.default_rng(n)
    s = scenes.Scene()
    for k in range(3):
        s.add_mesh(scenes.random_triangles((1, 3, 200)[k], seed=k, sigma=0.2), None)
    empty = s.add_mesh(np.zeros((0, 4), np.float32), None)
    for i in range(n):
        if i % 4 == 3:
            s.add_instance(empty, _affine(rng))
        s.add_instance(int(rng.integers(3)), _affine(rng))
    rays = _random_rays(rng, 3000, -3, 3)
    hits = both(torch_cuda, s, rays)
    assert np.array_equal(hits.view(np.uint32), orc.OracleScene(s).trace(rays, brute=True).view(np.uint32))
    assert (hits.view(np.int32)[:, 2] >= 0).any()


@pytest.mark.parametrize("rays", [2000, 140000])
@pytest.mark.parametrize("form", ["flat", "point", "thin", "nan", "inf"])
def test_transforms_without_a_usable_inverse(torch_cuda, form, rays):
    rng = np.random.default_rng(len(form))
    s = scenes.Scene()
    m = s.add_mesh(scenes.random_triangles(200, seed=1, sigma=0.2), None)
    for i in range(30):
        T = np.array(_affine(rng), np.float64).reshape(4, 4)
        if i % 5 == 2:
            T[:3, :3] = {"flat": np.diag([1, 1, 0]), "point": np.zeros((3, 3)), "thin": np.diag([1, 1e-5, 1]),
                         "nan": np.full((3, 3), np.nan), "inf": np.diag([np.inf, 1, 1])}[form]
        s.add_instance(m, T.astype(np.float32).reshape(16))
    both(torch_cuda, s, _random_rays(rng, rays, -3, 3), loops=(0,))


def chain(n, factor, mid):
    """Triangles at distances factor^k: a tree about n / 2.5 levels deep."""
    base = np.array([[0, 0, 0], [0.1, 0, 0], [0, 0.1, 0.05]], np.float32)
    v = np.concatenate([(base + [1, 0.3, 0.2]) * float(factor) ** (k - mid) * (1 + 0.01 * j) for k in range(n) for j in range(5)])
    return np.column_stack([v, np.ones(len(v))]).astype(np.float32)


@pytest.mark.parametrize("blas,tlas,shrink", [(8, 100, 0), (60, 60, 0), (40, 100, 1), (100, 100, 0), (100, 60, 1), (150, 60, 0), (180, 40, 0), (100, 120, 1)])
def test_deep_trees(torch_cuda, blas, tlas, shrink):
    """Chains of instances of a chain: stacks of a wide node per binary level fit, fit only by the wide tree's own
    depth (40 of 100), and do not fit (100 of 100: fp32 nodes). The last is refused, as it was with a binary top level."""
    s = scenes.Scene()
    m = s.add_mesh(chain(blas, 2.0, blas // 2), None)
    for k in range(tlas):
        T = np.eye(4)
        T[:3, :3] *= 2.0 ** -(blas // 2 + 12) if shrink else 1
        T[:3, 3] = np.array([1.0, 0.4, 0.3]) * 1.9 ** (k - tlas // 2)
        s.add_instance(m, T.astype(np.float32).reshape(16))
    if tlas == 120:
        with pytest.raises(lh.LH2HIPError, match="too deep"):
            make_core(s, 1)
        return
    rng = np.random.default_rng(blas + tlas)
    rays = np.concatenate([_random_rays(rng, 1500, -f, f) for f in (1, 30, 1e4)])
    aim = np.array([1.0, 0.4, 0.3]) * rng.uniform(0.5, 3, (1500, 1)) * 2.0 ** rng.integers(-20, 20, (1500, 1))
    rays[:1500, 4:7] = (aim - rays[:1500, :3]) / np.linalg.norm(aim - rays[:1500, :3], axis=1, keepdims=True)
    both(torch_cuda, s, rays)
