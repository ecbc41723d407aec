"""Queries run on the caller's stream, scene updates and frames on the core's own:
an update that follows a query at once, queries on several streams and a query
beside a frame give what they give one after the other. Each query is held back
behind other work of its stream, so that it starts after the next call would."""
import numpy as np
import pytest

import lighthouse2_amd as lh
from lighthouse2_amd import scenes
from test_oracle import _affine, _random_rays

pytestmark = pytest.mark.gpu
TRIS, MANY = 20000, 140000           # MANY: more rays than a four-lane launch takes


def meshes():
    return [scenes.random_triangles(TRIS, seed=k, sigma=0.05) for k in (1, 2)]


def make(torch, two_level, refit, v):
    core = lh.RenderCore()
    core.Setting("refit", refit)
    core.SetGeometry(0, v)
    rng = np.random.default_rng(3)
    T = [_affine(rng) for _ in range(20)] if two_level else [np.eye(4)]
    for i, t in enumerate(T):
        core.SetInstance(i, 0, t)
    core.FinalizeInstances()
    return core


def held(torch, stream):
    """Work ahead of what comes next on the stream: some 20 ms."""
    with torch.cuda.stream(stream):
        a = torch.zeros((4096, 4096), device="cuda")
        for _ in range(24):
            a = a @ a


def launch(torch, core, stream, kind, rays):
    n = len(rays)
    out = torch.zeros((n, 4) if kind == "closest" else (n + 31) // 32, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    if kind != "plain":
        held(torch, stream)
    fn = core.trace_any if kind == "any" else core.trace_closest
    fn(rays.data_ptr(), out.data_ptr(), n, stream.cuda_stream)
    return out


@pytest.mark.parametrize("kind", ["closest", "any"])
@pytest.mark.parametrize("n", [3000, MANY])
@pytest.mark.parametrize("two_level", [False, True])
@pytest.mark.parametrize("update", ["rebuild", "refit", "move"])
@pytest.mark.parametrize("own", [True, False], ids=["own stream", "null stream"])
def test_update_after_query(torch_cuda, own, update, two_level, n, kind):
    torch = torch_cuda
    v = meshes()
    core = make(torch, two_level, int(update == "refit"), v[0])
    rays = torch.from_numpy(_random_rays(np.random.default_rng(n), n, -2, 2)).cuda()
    stream = torch.cuda.Stream() if own else torch.cuda.default_stream()
    assert own == (stream.cuda_stream != 0)
    want = launch(torch, core, torch.cuda.current_stream(), kind, rays)
    torch.cuda.synchronize()
    want = want.cpu()
    got = launch(torch, core, stream, kind, rays)
    assert not stream.query()                       # still to run
    if update == "move":
        core.SetInstance(0, 0, _affine(np.random.default_rng(9)))
    else:
        core.SetGeometry(0, v[1])
    core.FinalizeInstances()
    after = launch(torch, core, stream, kind, rays)
    torch.cuda.synchronize()
    assert torch.equal(got.cpu(), want)
    assert not torch.equal(after.cpu(), want)
    core.Shutdown()


@pytest.mark.parametrize("own", [True, False], ids=["own stream", "null stream"])
def test_update_after_bounce(torch_cuda, own):
    torch = torch_cuda
    v = meshes()
    core = make(torch, False, 0, v[0])
    rays = torch.from_numpy(_random_rays(np.random.default_rng(1), 5000)).cuda()
    hits = launch(torch, core, torch.cuda.current_stream(), "closest", rays).view(torch.float32)
    ids = torch.arange(len(rays), dtype=torch.int32, device="cuda")
    stream = torch.cuda.Stream() if own else torch.cuda.default_stream()

    def bounce():
        out, path, cnt = torch.zeros_like(rays), torch.zeros_like(ids), torch.zeros(1, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        held(torch, stream)
        core.bounce_diffuse(rays.data_ptr(), hits.data_ptr(), ids.data_ptr(), len(rays), 7, 1e-4, out.data_ptr(), path.data_ptr(), cnt.data_ptr(),
                            stream.cuda_stream)
        return out, path, cnt

    def ordered(o):
        torch.cuda.synchronize()
        n = int(o[2])
        k = torch.argsort(o[1][:n])
        return o[1][:n][k].cpu(), o[0][:n][k].view(torch.int32).cpu()

    want = ordered(bounce())
    late = bounce()
    assert not stream.query()
    core.SetGeometry(0, v[1])
    core.FinalizeInstances()
    got = ordered(late)
    assert len(want[0]) > 500 and all(torch.equal(a, b) for a, b in zip(got, want))
    core.Shutdown()


@pytest.mark.parametrize("late", [0, 1, 2])
def test_queries_on_several_streams(torch_cuda, late):
    """They share the ray feed and the stacks' overflow area; one of the streams is the null stream."""
    torch = torch_cuda
    core = make(torch, True, 0, meshes()[0])
    rays = [torch.from_numpy(_random_rays(np.random.default_rng(k), MANY, -2, 2)).cuda() for k in range(4)]
    want = []
    for r in rays:
        want.append(launch(torch, core, torch.cuda.current_stream(), "closest", r))
        torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.default_stream(), torch.cuda.Stream(), torch.cuda.default_stream()]
    out = [torch.zeros((MANY, 4), dtype=torch.int32, device="cuda") for _ in rays]
    torch.cuda.synchronize()
    held(torch, streams[late])                       # one late, the others at once
    for s, r, o in zip(streams, rays, out):
        core.trace_closest(r.data_ptr(), o.data_ptr(), MANY, s.cuda_stream)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(out, want))
    core.Shutdown()


@pytest.mark.parametrize("own", [True, False], ids=["own stream", "null stream"])
def test_query_beside_frames(torch_cuda, own):
    """A frame that is not waited for, and a query that still waits when a frame begins."""
    torch = torch_cuda
    s = scenes.cornell_box(sphere_tris=2000)
    core = lh.RenderCore()
    lh.load_scene(core, s)
    core.SetTarget(640, 400, 1)
    view = scenes.cornell_view(640, 400)
    rays = torch.from_numpy(_random_rays(np.random.default_rng(4), MANY, -2, 2)).cuda()
    stream = torch.cuda.Stream() if own else torch.cuda.default_stream()
    want = launch(torch, core, torch.cuda.current_stream(), "closest", rays)
    core.Render(view, lh.LH2_RESTART)
    image = core.read_image()
    late = launch(torch, core, stream, "closest", rays)
    assert not stream.query()
    core.Render(view, lh.LH2_RESTART, async_=True)
    beside = torch.zeros_like(late)
    core.trace_closest(rays.data_ptr(), beside.data_ptr(), MANY, torch.cuda.current_stream().cuda_stream)
    core.WaitForRender()
    torch.cuda.synchronize()
    assert torch.equal(late, want) and torch.equal(beside, want)
    assert np.array_equal(core.read_image().view(np.uint32), image.view(np.uint32))
    core.Shutdown()


def test_query_in_a_graph(torch_cuda):
    """A captured query (any size up to the four-lane limit) replays, and an update waits for the replays before it."""
    torch = torch_cuda
    v = meshes()
    core = make(torch, True, 0, v[0])
    rays = torch.from_numpy(_random_rays(np.random.default_rng(6), 3000, -2, 2)).cuda()
    want = launch(torch, core, torch.cuda.current_stream(), "closest", rays).clone()
    out = torch.zeros_like(want)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        core.trace_closest(rays.data_ptr(), out.data_ptr(), len(rays), torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        out.zero_()
        graph.replay()
        core.trace_closest(rays.data_ptr(), want.data_ptr(), len(rays), torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    out.zero_()
    held(torch, torch.cuda.current_stream())
    graph.replay()
    core.SetGeometry(0, v[1])
    core.FinalizeInstances()
    torch.cuda.synchronize()
    assert torch.equal(out, want)
    core.Shutdown()


def test_cleared_outputs_in_a_graph(torch_cuda):
    """An any-hit query and a bounce clear their outputs on every replay, with other work between the replays."""
    torch = torch_cuda
    core = make(torch, True, 0, meshes()[0])
    rays = torch.from_numpy(_random_rays(np.random.default_rng(8), 3001, -2, 2)).cuda()
    n = len(rays)
    want = launch(torch, core, torch.cuda.current_stream(), "any", rays).clone()
    hits = launch(torch, core, torch.cuda.current_stream(), "closest", rays).view(torch.float32)
    torch.cuda.synchronize()
    found = int((hits.view(torch.int32)[:, 2] >= 0).sum())
    mask, cnt = torch.zeros_like(want), torch.zeros(1, dtype=torch.int32, device="cuda")
    ids = torch.arange(n, dtype=torch.int32, device="cuda")
    out, path = torch.zeros((n + 50, 8), device="cuda"), torch.zeros(n + 50, dtype=torch.int32, device="cuda")   # room for a count that was not cleared
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        s = torch.cuda.current_stream().cuda_stream
        core.trace_any(rays.data_ptr(), mask.data_ptr(), n, s)
        core.bounce_diffuse(rays.data_ptr(), hits.data_ptr(), ids.data_ptr(), n, 7, 1e-4, out.data_ptr(), path.data_ptr(), cnt.data_ptr(), s)
    for k in range(5):
        mask.fill_(-1), cnt.fill_(50)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(mask, want) and int(cnt) == found, k
        launch(torch, core, torch.cuda.current_stream(), "any", rays[: 100 + k])
    core.Shutdown()
