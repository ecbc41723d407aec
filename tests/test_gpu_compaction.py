"""Compaction of a wave's extension and shadow rays (one atomic per block of
256 paths; 512 rays for the bounce helper): frames whose path counts sit at
the edges of a block, and jobs whose paths share waves, against the oracle and
against the same jobs run alone. Every comparison is exact: path slots and random numbers
are keyed by the path's index, so no result depends on the order of the rays."""
import numpy as np
import pytest

import lighthouse2_amd as lh
from lighthouse2_amd import core as C
from lighthouse2_amd import scenes
import oracle as orc

pytestmark = pytest.mark.gpu
SIZES = [(1, 1), (255, 1), (16, 16), (257, 1), (127, 5)]


@pytest.mark.parametrize("w,h", SIZES)
@pytest.mark.parametrize("estimator", [0, 1])
def test_block_edges_match_oracle(torch_cuda, w, h, estimator):
    s = scenes.cornell_box(sphere_tris=400)
    view = scenes.cornell_view(w, h)
    core = lh.RenderCore()
    lh.load_scene(core, s)
    core.SetTarget(w, h, 1)
    for k, v in (("estimator", estimator), ("epsilon", 1e-3), ("maxDepth", 3)):
        core.Setting(k, v)
    core.Render(view, lh.LH2_RESTART)
    acc = core.read_accumulator_f64()
    core.Shutdown()
    if estimator == 0:
        ref = orc.render(s, view, w, h, 1, 1, 3, 1e-3, modes=[orc.RESTART])[1]
    else:
        ref = orc.render7(s, view, w, h, 1, 1, threads=4, modes=[orc.RESTART])[1]
    assert np.array_equal(acc, ref)


@pytest.mark.parametrize("sizes", [[(1, 1)] * 16, [(13, 5), (64, 1), (1, 3), (31, 9)], [(255, 1), (257, 1)]])
def test_jobs_sharing_waves_equal_jobs_alone(torch_cuda, sizes):
    """Job boundaries inside a wave: lanes of several jobs in one wavefront."""
    s = scenes.cornell_box(sphere_tris=400)
    core = lh.RenderCore()
    lh.load_scene(core, s)
    core.Setting("estimator", 1)
    server = lh.RenderServer(core)
    server.pause()
    ids = [server.submit(scenes.cornell_view(w, h), w, h, 2, 3, 77 + k) for k, (w, h) in enumerate(sizes)]
    server.pause(False)
    images = []
    for i in ids:
        server.wait(i, 60.0)
        images.append(server.read(i))
    assert server.stats()["max_parts"] == len(sizes)
    for k, ((w, h), img) in enumerate(zip(sizes, images)):
        i = server.submit(scenes.cornell_view(w, h), w, h, 2, 3, 77 + k)
        server.wait(i, 60.0)
        assert np.array_equal(server.read(i), img), (w, h)
    server.close()
    core.Shutdown()


@pytest.mark.parametrize("n", [1, 63, 511, 512, 513, 1500])
def test_bounce_block_edges(torch_cuda, n):
    torch = torch_cuda
    s = scenes.random_triangle_scene(3000, seed=5)
    core = lh.RenderCore()
    lh.load_scene(core, s)
    rays = orc.primary_rays(scenes.microbench_view(40, 40), 40, 40, 1234, 1e-5)[:n]
    o = orc.OracleScene(s)
    pid = np.arange(n, dtype=np.uint32)
    want, want_id = o.bounce(rays, o.trace(rays), pid, 91771, 1e-5)
    r = torch.from_numpy(np.ascontiguousarray(rays)).cuda()
    h, r2 = torch.zeros((n, 4), device="cuda"), torch.zeros((n, 8), device="cuda")
    p, p2, k = torch.arange(n, dtype=torch.int32, device="cuda"), torch.zeros(n, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    core.trace_closest(r.data_ptr(), h.data_ptr(), n)
    core.bounce_diffuse(r.data_ptr(), h.data_ptr(), p.data_ptr(), n, 91771, 1e-5, r2.data_ptr(), p2.data_ptr(), k.data_ptr())
    torch.cuda.synchronize()
    m = int(k.item())
    assert m == len(want)
    order = np.argsort(p2.cpu().numpy()[:m])
    assert np.array_equal(p2.cpu().numpy()[:m][order].astype(np.uint32), np.sort(want_id))
    assert np.array_equal(r2.cpu().numpy()[:m][order].view(np.uint32), want[np.argsort(want_id)].view(np.uint32))
    core.Shutdown()


@pytest.mark.parametrize("w,h,spp", [(362, 363, 1), (5, 26300, 1), (131100, 1, 1), (181, 363, 2)])
@pytest.mark.parametrize("estimator", [0, 1])
def test_tile_order_covers_every_path(torch_cuda, w, h, spp, estimator):
    """Frames of more than 131,072 paths start in tiles of 8 x 4 pixels: ragged widths and last bands, an image narrower
    than a tile, a band longer than the image, bands across two samples."""
    s = scenes.cornell_box(sphere_tris=400)
    view = scenes.cornell_view(w, h)
    core = lh.RenderCore()
    lh.load_scene(core, s)
    core.SetTarget(w, h, spp)
    for k, v in (("estimator", estimator), ("epsilon", 1e-3), ("maxDepth", 3)):
        core.Setting(k, v)
    core.Render(view, lh.LH2_RESTART)
    acc = core.read_accumulator_f64()
    core.Shutdown()
    if estimator == 0:
        ref = orc.render(s, view, w, h, spp, 1, 3, 1e-3, modes=[orc.RESTART])[1]
    else:
        ref = orc.render7(s, view, w, h, spp, 1, threads=16, modes=[orc.RESTART])[1]
    assert np.array_equal(acc, ref)
