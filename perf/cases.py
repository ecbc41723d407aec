"""What RenderCore_HIP is measured on: ray queries, scene updates, frames, served
jobs, and the two denoisers, each through the package's public entry points.

`listed()` names the cases, `draw(rng)` gives more of the same ranges. `prepare`
makes what a program holds before the call (scene, rays, handles, weights),
`run` is one pass, `exact` the same outputs in 64 bits by plain torch where such
a computation exists (a brute-force ray query, the U-Net and its gradients)."""
import copy
import functools
import math

import numpy as np
import torch

import lighthouse2_amd as lh
from lighthouse2_amd import scenes
from lighthouse2_amd import denoiser as dn

DEV = "cuda"


def listed():
    return [
        # picking / visibility probes of an editor: a few thousand rays against a mid-size mesh, latency counts
        {"name": "query_small", "kind": "query", "scene": "soup", "tris": 20000, "rays": 4096, "any": False},
        # ambient-occlusion baking: incoherent rays from the surface of the benchmark's 4M-triangle scene
        {"name": "bake_incoherent", "kind": "query", "scene": "soup", "tris": 4000000, "rays": 1999993, "any": False},
        # shadow rays towards area lights over an instanced scene (two-level tree, any hit, bit mask out)
        {"name": "shadow_instanced", "kind": "query", "scene": "instanced", "tris": 100000, "rays": 1000001, "any": True},
        # loading or rebuilding a scanned-size mesh, then the first look at it
        {"name": "load_mesh", "kind": "load", "tris": 500000, "rays": 65536},
        # one animation step: a deformed mesh refitted, every instance moved, the top level rebuilt, a preview traced
        {"name": "animate", "kind": "animate", "tris": 40000, "instances": 1000, "rays": 65536},
        # the parity configuration: Cornell box, 16 converging frames of the reference estimator, read back once
        {"name": "converge_cornell", "kind": "converge", "estimator": 0, "w": 256, "h": 256, "spp": 1, "frames": 16},
        # an interactive session at 1080p: filter estimator + SVGF + TAA, the camera moves every frame, a screenshot at the end
        {"name": "session_1080p", "kind": "session", "w": 1920, "h": 1080, "frames": 8},
        # a burst of preview and still jobs through the job server: optix7 stills, SVGF and learned denoising
        {"name": "serve_burst", "kind": "serve", "w": 512, "h": 384, "spp": 4, "jobs": 12},
        # SVGF on another renderer's 1080p G-buffer, moving camera
        {"name": "svgf_1080p", "kind": "svgf", "w": 1920, "h": 1080, "taa": True},
        # learned denoising of a 1080p frame (padded to 1088 rows)
        {"name": "denoise_1080p", "kind": "denoise", "w": 1920, "h": 1080},
        # one optimiser step of denoiser training on a 256x256 pair, the size it is trained at
        {"name": "train_256", "kind": "train", "w": 256, "h": 256},
        # the same step on whole 1080p frames
        {"name": "train_1080p", "kind": "train", "w": 1920, "h": 1088},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["query", "query", "load", "animate", "converge", "session", "serve", "svgf", "denoise", "train"])
    if kind == "query":
        if rng.random() < 0.6:
            return {"kind": "query", "scene": "soup", "tris": _log(rng, 1000, 3000000), "rays": _log(rng, 1000, 1900000), "any": rng.random() < 0.4}
        return {"kind": "query", "scene": "instanced", "tris": _log(rng, 20000, 100000), "rays": _log(rng, 1000, 1000000), "any": rng.random() < 0.5}
    if kind == "load":
        return {"kind": "load", "tris": _log(rng, 1000, 480000), "rays": _log(rng, 4096, 65536)}
    if kind == "animate":
        return {"kind": "animate", "tris": _log(rng, 2000, 40000), "instances": _log(rng, 20, 990), "rays": _log(rng, 4096, 65536)}
    if kind == "converge":
        return {"kind": "converge", "estimator": rng.choice([0, 1]), "w": _log(rng, 64, 400), "h": _log(rng, 64, 400), "spp": rng.choice([1, 2, 4]),
                "frames": rng.randint(1, 4)}
    if kind == "session":
        return {"kind": "session", "w": _log(rng, 320, 1900), "h": _log(rng, 200, 1070), "frames": rng.randint(1, 7)}
    if kind == "serve":
        return {"kind": "serve", "w": _log(rng, 96, 500), "h": _log(rng, 96, 380), "spp": rng.choice([1, 2, 4]), "jobs": rng.randint(1, 11)}
    if kind == "svgf":
        return {"kind": "svgf", "w": _log(rng, 101, 1919), "h": _log(rng, 75, 1079), "taa": rng.random() < 0.5}
    if kind == "denoise":
        return {"kind": "denoise", "w": _log(rng, 100, 1919), "h": _log(rng, 64, 1079)}
    return {"kind": "train", "w": 16 * _log(rng, 4, 120), "h": 16 * _log(rng, 4, 66)}


# ---- scenes -----------------------------------------------------------------
def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1000003 + salt)


def _soup(n, seed):
    """Random triangles as the incoherent benchmark has them: centroids uniform in the unit cube, vertex offsets of the mean spacing."""
    g = _gen(seed, 1)
    c = torch.rand((n, 1, 3), generator=g, device=DEV)
    v = torch.ones((n, 3, 4), device=DEV)
    v[:, :, :3] = c + torch.randn((n, 3, 3), generator=g, device=DEV) * (0.794 / n ** (1 / 3))
    return v


@functools.lru_cache(maxsize=4)
def _assets(meshes, tris, tex_size, lights):
    """Meshes, textures, materials and lights of the instanced workload: a program has these on disk."""
    return scenes.instanced_scene(meshes=meshes, tris=(tris // 2, tris), instances=0, tex_size=tex_size, lights=lights)


def _instanced(tris, instances, seed, tex_size=1024, lights=64):
    """The instanced workload (displaced spheres, textured, Disney materials, area lights) with this seed's placement."""
    base = _assets(6, tris, tex_size, lights)
    s = copy.copy(base)
    rng = np.random.default_rng(seed)
    s.instances = list(base.instances)         # the lights' instance stays first: its triangles refer to it
    for _ in range(instances):
        q = rng.normal(size=4)
        w, x, y, z = q / np.linalg.norm(q)
        R = np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)],
                      [2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)],
                      [2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]])
        M = np.eye(4)
        M[:3, :3] = R * rng.uniform(0.5, 2.0)
        M[:3, 3] = rng.uniform(-50, 50, 3)
        s.instances.append((int(rng.integers(0, 6)), M.reshape(16).astype(np.float32)))
    return s


def _rays(o, d, tmin, tmax):
    r = torch.empty((len(o), 8), device=DEV)
    r[:, 0:3], r[:, 3], r[:, 4:7], r[:, 7] = o, tmin, d, tmax
    return r.contiguous()


def _camera_rays(view, n, seed):
    """About n rays through a pinhole view, row by row, jittered."""
    g = _gen(seed, 5)
    w = int(math.ceil(math.sqrt(n)))
    i = torch.arange(n, device=DEV)
    p1, p2, p3, pos = (torch.tensor(np.asarray(view[k][0], np.float32), device=DEV) for k in ("p1", "p2", "p3", "pos"))
    u = ((i % w) + torch.rand(n, generator=g, device=DEV)) / w
    v = ((i // w) + torch.rand(n, generator=g, device=DEV)) / w
    d = p1 + u[:, None] * (p2 - p1) + v[:, None] * (p3 - p1) - pos
    return _rays(pos.expand(n, 3), torch.nn.functional.normalize(d, dim=1), 1e-4, 1e30)


def _bake_rays(v, n, seed):
    """Ambient-occlusion rays: points on the triangles in the order of a spatial grid, cosine-distributed about the surface normal, of finite length."""
    g = _gen(seed, 2)
    t = v[torch.randint(0, len(v), (n,), generator=g, device=DEV), :, :3]
    cell = (t.mean(1) * 64).clamp(0, 63).long()
    t = t[torch.argsort((cell[:, 2] * 64 + cell[:, 1]) * 64 + cell[:, 0], stable=True)]
    a, b = torch.rand(n, 1, generator=g, device=DEV).sqrt(), torch.rand(n, 1, generator=g, device=DEV)
    P = t[:, 0] * (1 - a) + t[:, 1] * (a * (1 - b)) + t[:, 2] * (a * b)
    N = torch.nn.functional.normalize(torch.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0], dim=1), dim=1)
    N = N * (torch.randint(0, 2, (n, 1), generator=g, device=DEV) * 2 - 1)
    S = torch.nn.functional.normalize(torch.randn(n, 3, generator=g, device=DEV), dim=1)
    return _rays(P + 1e-4 * N, torch.nn.functional.normalize(N * 1.001 + S, dim=1), 1e-5, 2.0)


def _surface_rays(s, n, seed, shadow):
    """From points on the instances' surfaces: to the area lights (shadow), or in cosine-distributed directions."""
    rng = np.random.default_rng(seed + 17)
    inst = np.sort(rng.integers(1, len(s.instances), n))
    o, nrm = np.empty((n, 3), np.float32), np.empty((n, 3), np.float32)
    mesh = np.array([m for m, _ in s.instances])
    T = np.stack([t.reshape(4, 4) for _, t in s.instances]).astype(np.float32)
    for m in range(6):
        k = np.nonzero(mesh[inst] == m)[0]
        v = s.meshes[m][0].reshape(-1, 3, 4)[:, :, :3]
        t = v[rng.integers(0, len(v), len(k))]
        b = rng.dirichlet((1, 1, 1), len(k)).astype(np.float32)
        R = T[inst[k]]
        P = (t * b[:, :, None]).sum(1)
        N = np.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0])
        N *= np.where((N * P).sum(1) < 0, -1, 1)[:, None]
        o[k] = np.einsum("nij,nj->ni", R[:, :3, :3], P) + R[:, :3, 3]
        N = np.einsum("nij,nj->ni", R[:, :3, :3], N)
        nrm[k] = N / np.maximum(np.linalg.norm(N, axis=1, keepdims=True), 1e-20)
    o += 1e-3 * nrm
    if shadow:
        L = s.tri_lights["centre"].astype(np.float32)[rng.integers(0, len(s.tri_lights), n)]
        d = L - o
        dist = np.linalg.norm(d, axis=1, keepdims=True)
        return _rays(torch.tensor(o, device=DEV), torch.tensor(d / dist, device=DEV), 1e-4, torch.tensor(dist[:, 0] - 2e-3, device=DEV))
    S = rng.normal(size=(n, 3)).astype(np.float32)
    d = nrm * 1.001 + S / np.linalg.norm(S, axis=1, keepdims=True)
    return _rays(torch.tensor(o, device=DEV), torch.tensor(d / np.linalg.norm(d, axis=1, keepdims=True), device=DEV), 1e-4, 1e30)


@functools.lru_cache(maxsize=8)
def _sphere(n, shape):
    """A displaced sphere of about n triangles with its CoreTri records."""
    a, b, c, _ = scenes.displaced_sphere(n, 1.0, seed=shape)
    return scenes.add_triangles(a, b, c, 0)


def _stretched(n, seed):
    """The sphere, stretched by this seed: another mesh of the same topology."""
    v, t = _sphere(n, seed % 2)
    k = np.random.default_rng(seed).uniform(0.7, 1.3, 4).astype(np.float32)
    k[3] = 1
    return np.ascontiguousarray(v * k), t


def _look(seed, w, h, extent=50.0):
    """A camera outside the cloud of instances, looking at a point inside it."""
    rng = np.random.default_rng(seed + 3)
    a = rng.uniform(0, 2 * np.pi)
    pos = np.array([2.4 * extent * np.sin(a), rng.uniform(0.1, 0.4) * extent, 2.4 * extent * np.cos(a)])
    at = rng.uniform(-0.1, 0.1, 3) * extent
    return pos, at, lambda k: scenes.camera_view(pos + (at - pos) * 0.002 * k, at, 45.0, w, h)


# ---- denoiser inputs ----------------------------------------------------------
def _params(seed):
    """He-normal weights, small random biases; the padding channels unused, as the trained network has them."""
    rng = np.random.default_rng(seed)
    p = {}
    for name, ci, co in dn.layer_specs():
        w = (rng.standard_normal((9, co, ci)) * math.sqrt(2.0 / (9 * ci))).astype(np.float32)
        b = (rng.standard_normal(co) * 0.02).astype(np.float32)
        if name == "e1_0":
            w[:, :, 10:] = 0
        if name == "out":
            w, b = w * np.float32(0.25), b + np.float32(0.8)     # log radiance: positive, as a trained network's
            w[:, 3:], b[3:] = 0, 0
        p[name] = (w, b)
    return p


def _frame(w, h, seed):
    """A noisy 1-spp frame of two textured planes with its packed G-buffer, and the next camera."""
    x = 0.005 * (seed % 7)
    v0 = scenes.camera_view((0.5 + x, 0.6, -1.0), (0.5, 0.5, 1.0), 50.0, w, h)
    v1 = scenes.camera_view((0.505 + x, 0.6, -0.999), (0.5, 0.5, 1.0), 50.0, w, h)
    acc, feat, wp, dd = scenes.gbuffer(v0, w, h, seed=seed)
    return [torch.from_numpy(np.ascontiguousarray(a)).to(DEV) for a in (acc, feat.view(np.int32), wp, dd)], v1


def _pair(w, h, seed):
    """A training pair in the network's terms: demodulated log radiance, albedo, normal, depth; and a clean target."""
    g = _gen(seed, 9)
    y, x = torch.meshgrid(torch.arange(h, device=DEV) / h, torch.arange(w, device=DEV) / w, indexing="ij")
    base = torch.stack([torch.sin(9 * x + 3 * y), torch.cos(7 * y - 2 * x), torch.sin(5 * (x + y)), torch.ones_like(x)], -1) * 0.4 + 0.6
    rad = torch.log1p(base * -torch.log(torch.rand((h, w, 1), generator=g, device=DEV).clamp_min(1e-6)))
    alb = (base * 0.8 + 0.1 * torch.rand((h, w, 4), generator=g, device=DEV)).clamp(0, 1)
    nrm = torch.nn.functional.normalize(torch.randn((h, w, 4), generator=g, device=DEV) * 0.1 + torch.tensor([0, 0, 1.0, 0], device=DEV), dim=-1)
    dep = torch.log1p(2 + x + 3 * y) * 0.1
    return [t.float().contiguous() for t in (rad, alb, nrm, dep)], torch.log1p(base).float().contiguous()


# ---- prepare --------------------------------------------------------------------
def _core(s):
    core = lh.RenderCore()
    lh.load_scene(core, s)
    return core


def prepare(case, seed):
    kind = case["kind"]
    if kind == "query":
        n = case["rays"]
        if case["scene"] == "soup":
            v = _soup(case["tris"], seed)
            core = lh.RenderCore()
            core.SetGeometry(0, v.reshape(-1, 4).cpu().numpy())
            core.SetInstance(0, 0, np.eye(4))
            core.FinalizeInstances()
            rays = _bake_rays(v, n, seed)
        else:
            s = _instanced(case["tris"], 1000, seed)
            core, rays = _core(s), _surface_rays(s, n, seed, case["any"])
        out = torch.zeros((n + 31) // 32, dtype=torch.int32, device=DEV) if case["any"] else torch.zeros((n, 4), device=DEV)
        return {"kind": "any" if case["any"] else "closest", "core": core, "rays": rays, "out": out}
    if kind == "load":
        v, t = _stretched(case["tris"], seed)
        view = scenes.camera_view((0.3, 0.5, -3.0), (0.0, 0.0, 0.0), 45.0, 256, 256)
        core = lh.RenderCore()
        core.SetMaterials(lh.formats.lambert_material((0.6, 0.5, 0.4)))
        return {"kind": kind, "core": core, "verts": v, "tris": t, "rays": _camera_rays(view, case["rays"], seed),
                "out": torch.zeros((case["rays"], 4), device=DEV)}
    if kind == "animate":
        s = _instanced(40000, case["instances"], seed, tex_size=256)
        v, t = _stretched(case["tris"], seed)
        bend = lambda k: np.ascontiguousarray(v + np.float32(0.05) * np.sin(v[:, [1, 2, 0, 3]] * 3 + k).astype(np.float32) * np.float32([1, 1, 1, 0]))
        rng = np.random.default_rng(seed)
        move = rng.uniform(-0.5, 0.5, (len(s.instances), 3)).astype(np.float32)
        steps = [[(i, m, _moved(T, move[i] * k)) for i, (m, T) in enumerate(s.instances) if i] for k in (0, 1)]
        core = _core(s)
        core.Setting("refit", 1)
        core.SetGeometry(0, v, t)
        core.FinalizeInstances()
        _, _, view = _look(seed, 256, 256)
        return {"kind": kind, "core": core, "poses": [bend(0), bend(1)], "tris": t, "steps": steps, "frame": 0,
                "rays": _camera_rays(view(0), case["rays"], seed), "out": torch.zeros((case["rays"], 4), device=DEV)}
    if kind == "converge":
        s = scenes.cornell_box(seed=seed) if case["estimator"] == 0 else scenes.disney_cornell_box(seed=seed)
        core = _core(s)
        core.SetTarget(case["w"], case["h"], case["spp"])
        for k, v in (("estimator", case["estimator"]), ("maxDepth", 3), ("epsilon", 1e-3)):
            core.Setting(k, v)
        return {"kind": kind, "core": core, "view": scenes.cornell_view(case["w"], case["h"]), "frames": case["frames"]}
    if kind == "session":
        core = _core(_instanced(100000, 1000, seed))
        core.SetTarget(case["w"], case["h"], 1)
        core.Setting("estimator", 2)
        _, _, view = _look(seed, case["w"], case["h"])
        return {"kind": kind, "core": core, "views": [view(k) for k in range(case["frames"])]}
    if kind == "serve":
        core = _core(_instanced(40000, 300, seed, tex_size=512, lights=16))
        core.Setting("estimator", 1)
        server = lh.RenderServer(core, budget_bytes=8 << 30, pass_paths=1 << 22)
        server.set_denoiser(dn.UNetDenoiser(16, 16, params=_params(seed)).weights_blob())
        rng = np.random.default_rng(seed)
        jobs = []
        for k in range(case["jobs"]):     # whole sizes and halves; plain stills take four times the samples of denoised ones
            w, h = (case["w"], case["h"]) if k % 3 != 1 else ((case["w"] + 1) // 2, (case["h"] + 1) // 2)
            denoise = k % 3
            jobs.append((_look(int(rng.integers(1 << 20)), w, h)[2](0), w, h, case["spp"] * (1 if denoise else 4), 3, int(rng.integers(1, 1 << 24)), denoise))
        return {"kind": kind, "server": server, "jobs": jobs}
    if kind == "svgf":
        frame, view = _frame(case["w"], case["h"], seed)
        return {"kind": kind, "svgf": lh.Svgf(case["w"], case["h"], taa=case["taa"]), "frame": frame, "view": view,
                "out": torch.zeros((case["h"], case["w"], 4), device=DEV)}
    if kind == "denoise":
        w, h = case["w"], case["h"]
        frame, _ = _frame(w, h, seed)
        net = dn.UNetDenoiser((h + 15) // 16 * 16, (w + 15) // 16 * 16, params=_params(seed))
        return {"kind": kind, "net": net, "acc": frame[0], "feat": frame[1], "w": w, "h": h, "out": torch.zeros((h, w, 4), device=DEV)}
    net = dn.UNetDenoiser(case["h"], case["w"], params=_params(seed))
    inputs, target = _pair(case["w"], case["h"], seed)
    return {"kind": kind, "net": net, "inputs": inputs, "target": target}


def _moved(T, d):
    M = T.reshape(4, 4).copy()
    M[:3, 3] += d
    return M.reshape(16)


# ---- run --------------------------------------------------------------------------
def _hits(core, rays, out):
    core.trace_closest(rays.data_ptr(), out.data_ptr(), len(rays), torch.cuda.current_stream().cuda_stream)
    return {"ids": out.view(torch.int32)[:, :3], "t": out[:, 3]}


def run(st):
    kind = st["kind"]
    if kind == "closest":
        return _hits(st["core"], st["rays"], st["out"])
    if kind == "any":
        st["core"].trace_any(st["rays"].data_ptr(), st["out"].data_ptr(), len(st["rays"]), torch.cuda.current_stream().cuda_stream)
        return st["out"]
    if kind == "load":
        core = st["core"]
        core.SetGeometry(0, st["verts"], st["tris"])
        core.SetInstance(0, 0, np.eye(4))
        core.FinalizeInstances()
        return _hits(core, st["rays"], st["out"])
    if kind == "animate":
        core, k = st["core"], st["frame"]
        st["frame"] = 1 - k
        core.SetGeometry(0, st["poses"][k], st["tris"])
        for i, m, T in st["steps"][k]:
            core.SetInstance(i, m, T)
        core.FinalizeInstances()
        return _hits(core, st["rays"], st["out"])
    if kind == "converge":
        core = st["core"]
        for k in range(st["frames"]):
            core.Render(st["view"], lh.LH2_RESTART if k == 0 else lh.LH2_CONVERGE)
        return {"image": core.read_image(), "sums": core.read_accumulator_f64()}
    if kind == "session":
        core = st["core"]
        for v in st["views"]:
            core.Render(v, lh.LH2_RESTART)
        return core.read_image()
    if kind == "serve":
        server = st["server"]
        ids = [server.submit(v, w, h, spp, depth, seed, denoise=d) for v, w, h, spp, depth, seed, d in st["jobs"]]
        images = []
        for i in ids:
            server.wait(i)
            images.append(server.read(i))
        return images
    if kind == "svgf":
        acc, feat, wp, dd = st["frame"]
        st["svgf"].frame(acc.data_ptr(), feat.data_ptr(), wp.data_ptr(), dd.data_ptr(), st["view"], st["out"].data_ptr(), j=(0.1, -0.1),
                         stream=torch.cuda.current_stream().cuda_stream)
        return st["out"]
    net = st["net"]
    if kind == "denoise":
        net.denoise_frame(st["acc"], st["feat"], 1, st["w"], st["h"], st["out"])
        return st["out"]
    net.set_input(*st["inputs"])
    out = net.forward()
    loss = net.loss_backward(st["target"])
    net.step(lr=2e-3)
    return {"out": out, "loss": loss, "layers": [(d["gw"], d["gb"], d["w"]) for d in net.p.values()]}


# ---- work -------------------------------------------------------------------------
def _conv_flops(w, h):
    return sum(18 * ci * co * (h >> lvl) * (w >> lvl) for name, ci, co in dn.layer_specs() for lvl in [0 if name == "out" else int(name.split("_")[1])])


def work(case):
    kind = case["kind"]
    if kind == "query":
        n, t = case["rays"], case["tris"] * (1 if case["scene"] == "soup" else 5)
        return {"bytes": n * (32 + (0.125 if case["any"] else 16)) + min(t, 32 * n) * (36 + 16), "flops": 0}
    if kind == "load":     # vertices and records in, tree and leaf triangles out, rays and hits
        return {"bytes": case["tris"] * (48 + 208 + 48 + 24) + case["rays"] * 48, "flops": 0}
    if kind == "animate":
        return {"bytes": case["tris"] * (48 + 208 + 48 + 24) + case["instances"] * (64 + 128) + case["rays"] * 48, "flops": 0}
    px = case["w"] * case["h"]
    if kind == "converge":   # per sample a hit, a record, a material and a contribution; 32- and 64-bit sums per frame; the image once
        return {"bytes": px * (case["frames"] * (case["spp"] * 2 * (16 + 128) + 96) + 48), "flops": 0}
    if kind == "session":    # two vertices per path, the G-buffer, the sums, SVGF's inputs, history and image
        return {"bytes": px * (case["frames"] * (2 * (16 + 128 + 32) + 48 + 96 + 200) + 16), "flops": 0}
    if kind == "serve":
        return {"bytes": sum(px * (4 * case["spp"] * 288 if k % 3 == 0 else (0.25 if k % 3 == 1 else 1) * (case["spp"] * 352 + 300)) for k in range(case["jobs"])), "flops": 0}
    if kind == "svgf":       # accumulators, features, positions and derivatives in, history in and out, image out
        return {"bytes": px * (32 + 48 + 2 * (16 + 16 + 16) + 16 + (32 if case["taa"] else 0)), "flops": px * 3 * 20 * 60}
    if kind == "denoise":
        return {"bytes": px * (32 + 16 + 16), "flops": _conv_flops((case["w"] + 15) // 16 * 16, (case["h"] + 15) // 16 * 16)}
    # training: every activation is written by the forward and read by the backward pass (64 + 32 channels of bf16 per pixel and level)
    return {"bytes": px * (52 + 64 + 16 + 2 * 1.33 * 2 * 128), "flops": 3 * _conv_flops(case["w"], case["h"])}


def tolerance(case):
    # Hits, rendered images and the filtered frame are defined bit for bit: every path's random numbers are keyed by its
    # index, contributions are added in sample order, the box tests only prune, ties go to the smaller id.
    # The network keeps bf16 activations: an order of sums changes roundings, which travel through 19 layers and back.
    # Measured against 64 bits: display image 4e-4, gradients up to 5e-3; four times that.
    return {"denoise": {"rel": 1.5e-3}, "train": {"rel": 2e-2}}.get(case["kind"], "exact")


# ---- exact ------------------------------------------------------------------------
def _bf(x):
    return x.to(torch.bfloat16).double()


def _conv(x, w, b):
    """3x3 convolution of (H, W, Ci) by (9, Co, Ci) in 64 bits, as nine products."""
    H, W, _ = x.shape
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    y = b.expand(H, W, -1)
    for t in range(9):
        y = y + p[t // 3:t // 3 + H, t % 3:t % 3 + W] @ w[t].T
    return y


def _unet(x, p):
    conv = lambda name, v: _conv(v, *p[name])
    skip = []
    for lvl in range(5):
        x = torch.relu(conv(f"e2_{lvl}", torch.relu(conv(f"e1_{lvl}", x))))
        if lvl < 4:
            skip.append(x)
            x = (x[0::2, 0::2] + x[0::2, 1::2] + x[1::2, 0::2] + x[1::2, 1::2]) * 0.25
    for lvl in range(3, -1, -1):
        x = torch.cat([x.repeat_interleave(2, 0).repeat_interleave(2, 1), skip[lvl]], -1)
        x = torch.relu(conv(f"d2_{lvl}", torch.relu(conv(f"d1_{lvl}", x))))
    return conv("out", x)


def _master(seed):
    return {k: tuple(torch.from_numpy(a).to(DEV) for a in v) for k, v in _params(seed).items()}


def _exact_query(case, seed):
    v = _soup(case["tris"], seed)
    rays = _bake_rays(v, case["rays"], seed).double()
    v = v[:, :, :3].double()
    e1, e2 = v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
    n = torch.cross(e1, e2, dim=1)
    best = rays[:, 7].clone()
    for k in range(0, len(rays), 512):     # Moeller-Trumbore, every ray against every triangle
        o, d, lo, hi = rays[k:k + 512, 0:3], rays[k:k + 512, 4:7], rays[k:k + 512, 3:4], rays[k:k + 512, 7:8]
        det = -(d @ n.T)
        t = ((o @ n.T) - (v[:, 0] * n).sum(1)) / det
        # with s = o - v0: u = (s x d) . e2 / det and v = -(s x d) . e1 / det, in products of the coordinates
        q = torch.cross(o, d, dim=1)
        u = (q @ e2.T - d @ torch.cross(e2, v[:, 0], dim=1).T) / det
        w = -(q @ e1.T - d @ torch.cross(e1, v[:, 0], dim=1).T) / det
        ok = (u >= 0) & (w >= 0) & (u + w <= 1) & (t > lo) & (t < hi)
        best[k:k + 512] = torch.minimum(best[k:k + 512], torch.where(ok, t, hi).amin(1))
    return {"ids": None, "t": best}


def exact(case, seed):
    kind = case["kind"]
    if kind == "query" and case["scene"] == "soup" and not case["any"] and case["tris"] * case["rays"] <= 2e9:
        return _exact_query(case, seed)
    if kind == "denoise":
        w, h = case["w"], case["h"]
        (acc, feat, _, _), _ = _frame(w, h, seed)
        f = feat.long() & 0xffffffff
        alb = torch.stack([(f[..., 0] >> 22) / 1023.0, ((f[..., 0] >> 11) & 2047) / 2047.0, (f[..., 0] & 2047) / 2047.0], -1).double()
        nrm = torch.stack([((f[..., 1] >> s) & 1023) / 511.0 - 1 for s in (2, 12, 22)], -1).double()
        dep = torch.log1p(feat[..., 2].contiguous().view(torch.float32).double().clamp_max(1e4)) * 0.1
        rad = torch.log1p((acc[0] + acc[1])[..., :3].double().clamp_min(0) / alb.clamp_min(0.02))
        x = torch.zeros(((h + 15) // 16 * 16, (w + 15) // 16 * 16, 16), dtype=torch.float64, device=DEV)
        x[:h, :w, :10] = _bf(torch.cat([rad, alb, nrm, dep[..., None]], -1))
        with torch.no_grad():
            o = _unet(x, {k: (_bf(a), b.double()) for k, (a, b) in _master(seed).items()})[:h, :w, :3]
        img = torch.zeros((h, w, 4), dtype=torch.float64, device=DEV)
        img[..., :3] = (torch.expm1(o.clamp_min(0)) * alb.clamp_min(0.02)).sqrt().sqrt()
        return img
    if kind == "train" and case["w"] * case["h"] <= 300000:
        (rad, alb, nrm, dep), target = _pair(case["w"], case["h"], seed)
        x = torch.zeros((case["h"], case["w"], 16), dtype=torch.float64, device=DEV)
        x[..., :10] = _bf(torch.cat([rad[..., :3], alb[..., :3], nrm[..., :3], dep[..., None]], -1))
        p = {k: (_bf(a).requires_grad_(), b.double().requires_grad_()) for k, (a, b) in _master(seed).items()}
        out = _unet(x, p)
        t = target[..., :3].double()
        loss = ((out[..., :3] - t) ** 2 / (t * t + 0.01)).mean()
        loss.backward()
        return {"out": out.detach(), "loss": loss.detach().reshape(1), "layers": [(a.grad, b.grad, None) for a, b in p.values()]}
    return None
