"""The backward pass's fused and batched kernels against the separate calls they
replace (bit for bit) and the weight gradient against FP64, at the edges of
their tiles: 32-pixel segments and 8-row chunks of the weight gradient, 16-
and 32-pixel tiles of the convolutions, 256-element blocks of the Adam step."""
import ctypes

import numpy as np
import pytest

import lighthouse2_amd as lh
from lighthouse2_amd import denoiser as D
import denoiser_ref as R

pytestmark = pytest.mark.gpu


def dev(torch, a):
    return torch.from_numpy(D.bf16_bits(a).reshape(-1).copy()).cuda()


def empty(torch, n):
    return torch.full((n,), 0x7f7f, dtype=torch.int16, device="cuda")


def check_dw(torch, x, gy, gw, gb, terms):
    """fp32 sums of `terms` exact products: within 1e-5 of the largest sum (as the unbatched entry point's test)."""
    rgw, rgb = R.conv_dw(x, gy)
    assert np.max(np.abs(gw.cpu().numpy().reshape(rgw.shape) - rgw)) <= 1e-5 * np.max(np.abs(rgw)), terms
    assert np.max(np.abs(gb.cpu().numpy() - rgb)) <= 1e-5 * np.max(np.abs(rgb)) + 1e-6, terms


@pytest.mark.parametrize("H,W", [(1, 1), (2, 31), (7, 32), (8, 33), (9, 64), (17, 65), (70, 34)])
def test_weight_gradient_tile_edges(torch_cuda, H, W):
    torch = torch_cuda
    L = lh.library()
    sh = torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(H * 100 + W)
    for cin, cout in ((16, 32), (32, 32), (64, 32), (32, 16), (16, 16)):
        x, gy = R.bf16(rng.standard_normal((H, W, cin))), R.bf16(rng.standard_normal((H, W, cout)))
        dx, dgy = dev(torch, x), dev(torch, gy)
        ws = torch.zeros(int(L.lh2hip_dn_dw_workspace_bytes(cin, cout)) // 4, device="cuda")
        gw, gb = torch.full((9 * cout * cin,), 7.0, device="cuda"), torch.full((cout,), 7.0, device="cuda")
        assert L.lh2hip_dn_conv3x3_dw(dx.data_ptr(), cin, dgy.data_ptr(), cout, H, W, gw.data_ptr(), gb.data_ptr(), ws.data_ptr(), sh) == 0
        torch.cuda.synchronize()
        check_dw(torch, x, gy, gw, gb, (cin, cout, H, W))


def test_weight_gradient_batch_with_concatenation(torch_cuda):
    """A list of layers of different sizes; one reads its 64 inputs from the two halves of a concatenation."""
    torch = torch_cuda
    L = lh.library()
    sh = torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(3)
    rows, keep, checks = [], [], []
    for cin, cout, H, W, cat in ((16, 32, 40, 70, False), (64, 32, 22, 70, True), (32, 16, 8, 32, False), (64, 32, 6, 34, False), (32, 32, 1, 5, False)):
        gy = R.bf16(rng.standard_normal((H, W, cout)))
        coarse = None
        if cat:
            c, k = R.bf16(rng.standard_normal((H // 2, W // 2, 32))), R.bf16(rng.standard_normal((H, W, 32)))
            x, coarse, dx = R.upcat(c, k), dev(torch, c), dev(torch, k)
        else:
            x = R.bf16(rng.standard_normal((H, W, cin)))
            dx = dev(torch, x)
        dgy, gw, gb = dev(torch, gy), torch.full((9 * cout * cin,), 7.0, device="cuda"), torch.full((cout,), 7.0, device="cuda")
        keep += [dx, dgy, coarse]
        rows.append(D._Layer(dx.data_ptr(), coarse.data_ptr() if cat else None, dgy.data_ptr(), gw.data_ptr(), gb.data_ptr(), cin, cout, H, W))
        checks.append((x, gy, gw, gb))
    t = (D._Layer * len(rows))(*rows)
    need = int(L.lh2hip_dn_dw_batch_workspace_bytes(t, len(rows)))
    ws = torch.zeros(need // 4, device="cuda")
    assert L.lh2hip_dn_conv3x3_dw_batch(t, len(rows), ws.data_ptr(), need - 4, sh) != 0      # too small: refused on the host
    assert L.lh2hip_dn_conv3x3_dw_batch(t, len(rows), ws.data_ptr(), need, sh) == 0
    torch.cuda.synchronize()
    for k, (x, gy, gw, gb) in enumerate(checks):
        check_dw(torch, x, gy, gw, gb, k)
    t[0].Cin = 48
    assert int(L.lh2hip_dn_dw_batch_workspace_bytes(t, len(rows))) == 0


@pytest.mark.parametrize("H,W", [(2, 2), (6, 18), (22, 70), (202, 1930)])
def test_input_gradients_equal_their_parts(torch_cuda, H, W):
    """dx_relu, dx_cat and pool2_bwd_relu; 202 x 1930 runs the large tiles, ragged both ways."""
    torch = torch_cuda
    L = lh.library()
    sh = torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(W)
    bf = lambda *s: R.bf16(rng.standard_normal(s))
    n = H * W
    act = bf(H, W, 32)
    act[rng.random(act.shape) < 0.3] = 0
    dact = dev(torch, act)
    for cin in (16, 32):
        gy, w = dev(torch, bf(H, W, cin)), dev(torch, bf(9, 32, cin) * 0.2)
        want, got = empty(torch, n * 32), empty(torch, n * 32)
        assert L.lh2hip_dn_conv3x3(gy.data_ptr(), cin, w.data_ptr(), None, want.data_ptr(), 32, H, W, 0, sh) == 0
        assert L.lh2hip_dn_relu_bwd(dact.data_ptr(), want.data_ptr(), want.data_ptr(), n * 32, sh) == 0
        assert L.lh2hip_dn_conv3x3_dx_relu(gy.data_ptr(), cin, w.data_ptr(), dact.data_ptr(), got.data_ptr(), 32, H, W, sh) == 0
        assert torch.equal(want, got), cin
    w64, ac = dev(torch, bf(9, 64, 32) * 0.2), dev(torch, bf(H // 2, W // 2, 32))
    cat, skip, coarse = empty(torch, n * 64), empty(torch, n * 32), empty(torch, n * 8)
    assert L.lh2hip_dn_conv3x3(gy.data_ptr(), 32, w64.data_ptr(), None, cat.data_ptr(), 64, H, W, 0, sh) == 0
    assert L.lh2hip_dn_upcat_bwd(cat.data_ptr(), 32, 32, H, W, coarse.data_ptr(), skip.data_ptr(), sh) == 0
    assert L.lh2hip_dn_relu_bwd(ac.data_ptr(), coarse.data_ptr(), coarse.data_ptr(), n * 8, sh) == 0
    skip2, coarse2 = empty(torch, n * 32), empty(torch, n * 8)
    assert L.lh2hip_dn_conv3x3_dx_cat(gy.data_ptr(), w64.data_ptr(), ac.data_ptr(), coarse2.data_ptr(), skip2.data_ptr(), H, W, sh) == 0
    assert torch.equal(skip, skip2) and torch.equal(coarse, coarse2)
    out = empty(torch, n * 32)
    assert L.lh2hip_dn_pool2_bwd_relu(coarse.data_ptr(), skip.data_ptr(), dact.data_ptr(), 32, H, W, out.data_ptr(), sh) == 0
    assert L.lh2hip_dn_pool2_bwd(coarse.data_ptr(), 32, H, W, skip.data_ptr(), 1, sh) == 0
    assert L.lh2hip_dn_relu_bwd(dact.data_ptr(), skip.data_ptr(), skip.data_ptr(), n * 32, sh) == 0
    assert torch.equal(skip, out)
    assert L.lh2hip_dn_conv3x3_dx_relu(gy.data_ptr() + 2, 32, w64.data_ptr(), dact.data_ptr(), got.data_ptr(), 32, H, W, sh) != 0


def test_adam_batch_and_vector_loss_equal_the_single_calls(torch_cuda):
    torch = torch_cuda
    L = lh.library()
    sh = torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(9)
    f = lambda n: torch.from_numpy(rng.standard_normal(n).astype(np.float32)).cuda()
    rows, single = [], []
    for n, co, ci in ((9 * 16 * 16, 16, 16), (1, 0, 0), (255, 0, 0), (257, 0, 0), (9 * 32 * 64, 32, 64)) + ((32, 0, 0),) * 50:
        p, m, v, g = f(n), f(n), f(n).abs(), f(n)
        wf, wb = empty(torch, n), empty(torch, n)
        q = [t.clone() for t in (p, m, v, wf, wb)]
        rows.append((p, m, v, g, wf, wb, n, co, ci))
        conv = co > 0
        assert L.lh2hip_dn_adam(q[0].data_ptr(), q[1].data_ptr(), q[2].data_ptr(), g.data_ptr(), n, 1e-3, 0.9, 0.999, 1e-8, 3,
                                q[3].data_ptr() if conv else None, q[4].data_ptr() if conv else None, co, ci, sh) == 0
        single.append(q)
    t = (D._Tensor * len(rows))(*[D._Tensor(p.data_ptr(), m.data_ptr(), v.data_ptr(), g.data_ptr(), wf.data_ptr() if co else None,
                                            wb.data_ptr() if co else None, n, co, ci) for p, m, v, g, wf, wb, n, co, ci in rows])
    assert L.lh2hip_dn_adam_batch(t, len(rows), 1e-3, 0.9, 0.999, 1e-8, 3, sh) == 0
    torch.cuda.synchronize()
    for (p, m, v, g, wf, wb, n, co, ci), q in zip(rows, single):
        assert all(torch.equal(a, b) for a, b in zip((p, m, v, wf, wb), q)), n
    # the loss of 16 channels: aligned (vector) against one element off (scalar kernel); the sum over blocks is an atomic
    H, W = 33, 70
    o, tgt = rng.standard_normal((H * W * 16 + 1,)).astype(np.float32), f(H * W * 4)
    res = []
    for off in (0, 1):
        buf = torch.zeros(H * W * 16 + 4, device="cuda")
        buf[off:off + H * W * 16] = torch.from_numpy(o[:H * W * 16]).cuda()
        dout, loss = empty(torch, H * W * 16), torch.zeros(1, device="cuda")
        assert L.lh2hip_dn_relmse(buf.data_ptr() + 4 * off, 16, tgt.data_ptr(), H, W, dout.data_ptr(), loss.data_ptr(), sh) == 0
        res.append((dout.clone(), float(loss.item())))
    assert torch.equal(res[0][0], res[1][0]) and abs(res[0][1] - res[1][1]) <= 1e-5 * res[0][1]   # 10 block sums in any order


def test_batch_records_match_the_header():
    assert ctypes.sizeof(D._Layer) == 56 and ctypes.sizeof(D._Tensor) == 64


@pytest.mark.parametrize("H,W", [(514, 62), (256, 128), (258, 130), (1038, 546)])
def test_row_tiles_equal_small_tiles(torch_cuda, H, W):
    """Large images (4 rows x 16 or 32 pixels a wave; with 64 channels, blocks that
    walk several tiles at 1038 x 546), ragged or whole both ways, against crops of
    the same input at even corners through the 4 x 16 tiles, whose sums run over
    the taps and channels in the same order: bit for bit."""
    torch = torch_cuda
    L = lh.library()
    sh = torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(H + W)
    bf = lambda *s: R.bf16(rng.standard_normal(s))
    x64, x32, coarse = bf(H, W, 64), bf(H, W, 32), bf(H // 2, W // 2, 32)
    w64, w32, wg = dev(torch, bf(9, 32, 64) * 0.2), dev(torch, bf(9, 32, 32) * 0.2), dev(torch, bf(9, 64, 32) * 0.2)
    b = torch.from_numpy(rng.standard_normal(32).astype(np.float32)).cuda()

    def run(y0, y1, x0, x1):
        h, w = y1 - y0, x1 - x0
        cut = lambda t: dev(torch, np.ascontiguousarray(t[y0:y1, x0:x1]))
        half = dev(torch, np.ascontiguousarray(coarse[y0 // 2:y1 // 2, x0 // 2:x1 // 2]))
        a, s, out = cut(x64), cut(x32), [empty(torch, h * w * 32) for _ in range(4)]
        small = [empty(torch, h * w * 8) for _ in range(2)]
        assert L.lh2hip_dn_conv3x3(a.data_ptr(), 64, w64.data_ptr(), b.data_ptr(), out[0].data_ptr(), 32, h, w, 1, sh) == 0
        assert L.lh2hip_dn_conv3x3_cat(half.data_ptr(), s.data_ptr(), w64.data_ptr(), b.data_ptr(), out[1].data_ptr(), 32, h, w, 1, sh) == 0
        assert L.lh2hip_dn_conv3x3_pool(s.data_ptr(), 32, w32.data_ptr(), b.data_ptr(), out[2].data_ptr(), 32, h, w, small[0].data_ptr(), sh) == 0
        assert L.lh2hip_dn_conv3x3_dx_cat(s.data_ptr(), wg.data_ptr(), half.data_ptr(), small[1].data_ptr(), out[3].data_ptr(), h, w, sh) == 0
        torch.cuda.synchronize()
        return [t.reshape(h, w, 32) for t in out] + [t.reshape(h // 2, w // 2, 32) for t in small]

    full = run(0, H, 0, W)
    for y0 in sorted({0, (H // 32) * 16 - 10, H - 28}):
        for x0 in sorted({0, max((W // 64) * 32 - 10, 0), W - 28}):
            y1, x1 = min(y0 + 28, H), min(x0 + 28, W)
            part = run(y0, y1, x0, x1)
            t, l = (2 if y0 else 0), (2 if x0 else 0)
            e, r = y1 - y0 - (2 if y1 < H else 0), x1 - x0 - (2 if x1 < W else 0)
            for k, (f, p) in enumerate(zip(full, part)):
                q = 1 if k < 4 else 2
                assert torch.equal(f[(y0 + t) // q:(y0 + e) // q, (x0 + l) // q:(x0 + r) // q], p[t // q:e // q, l // q:r // q]), (k, y0, x0)


def test_replaced_tensors_are_the_ones_used(torch_cuda):
    """Entries of the network's dictionaries replaced by other tensors: a step does what it does after copying into the old ones."""
    torch = torch_cuda
    H, W = 32, 48
    rng = np.random.default_rng(12)
    f = lambda *s: torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda()
    inputs, target = (f(H, W, 4).abs(), f(H, W, 4).abs(), f(H, W, 4), f(H, W).abs()), f(H, W, 4)
    nets = [D.UNetDenoiser(H, W, seed=5) for _ in range(2)]
    old = []

    def put(net, at, key, value):
        if net is nets[0]:
            at[key].copy_(value.view(at[key].shape))
        else:
            old.append((at[key], at[key].clone()))
            at[key] = value.clone().view(at[key].shape)

    new = {}
    for name, ci, co in D.layer_specs():
        for k, shape in (("w", (9, co, ci)), ("b", (co,))):
            new[name, k] = f(*shape) * 0.1
            new[name, "m" + k], new[name, "v" + k], new[name, "g" + k] = f(*shape) * 0.01, f(*shape).abs() * 0.01, f(*shape)
    for net in nets:
        for (name, k), t in new.items():
            put(net, net.p[name], k, t)
        net._cast()
        for d in (net.a, net.g):
            for k in list(d):
                put(net, d, k, torch.zeros_like(d[k]))
        put(net, vars(net), "dout", torch.zeros_like(net.dout))
        net.set_input(*inputs)
        net.forward()
        net.loss_backward(target)
        net.step(lr=1e-2)
    torch.cuda.synchronize()
    for name, ci, co in D.layer_specs():
        for k in nets[0].p[name]:
            a, b = nets[0].p[name][k], nets[1].p[name][k]
            assert a == b if isinstance(a, int) else torch.equal(a, b), (name, k)
    assert all(torch.equal(t, was) for t, was in old)


def test_images_taller_than_a_grid(torch_cuda):
    """65,552 rows: pool2_bwd_relu equals its parts, and a training step runs."""
    torch = torch_cuda
    L = lh.library()
    sh = torch.cuda.current_stream().cuda_stream
    H, W = 65552, 16
    rng = np.random.default_rng(2)
    rnd = lambda n: dev(torch, R.bf16(rng.standard_normal(n)))
    for C, w in ((8, 2), (32, W)):
        dy, skip, act, out = rnd(H * w * C // 4), rnd(H * w * C), rnd(H * w * C), empty(torch, H * w * C)
        assert L.lh2hip_dn_pool2_bwd_relu(dy.data_ptr(), skip.data_ptr(), act.data_ptr(), C, H, w, out.data_ptr(), sh) == 0
        assert L.lh2hip_dn_pool2_bwd(dy.data_ptr(), C, H, w, skip.data_ptr(), 1, sh) == 0
        assert L.lh2hip_dn_relu_bwd(act.data_ptr(), skip.data_ptr(), skip.data_ptr(), H * w * C, sh) == 0
        assert torch.equal(out, skip), C
    net = D.UNetDenoiser(H, W, seed=1)
    f = lambda *s: torch.rand(s, device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    before = net.p["e1_0"]["w"].clone()
    net.set_input(f(H, W, 4), f(H, W, 4), f(H, W, 4), f(H, W))
    net.forward()
    loss = net.loss_backward(f(H, W, 4))
    net.step()
    assert torch.isfinite(loss).all() and not torch.equal(net.p["e1_0"]["w"], before) and torch.isfinite(net.p["e1_0"]["w"]).all()


@pytest.mark.parametrize("H,W", [(161, 250), (163, 250), (521, 250), (527, 258)])
def test_weight_gradient_chunk_heights(torch_cuda, H, W):
    """Sizes whose chunks are 4 and 8 rows high (2 in the tests above), with a short last chunk."""
    torch = torch_cuda
    L = lh.library()
    sh = torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(H)
    for cin, cout in ((32, 32), (64, 32), (16, 16)):
        x, gy = R.bf16(rng.standard_normal((H, W, cin))), R.bf16(rng.standard_normal((H, W, cout)))
        dx, dgy = dev(torch, x), dev(torch, gy)
        ws = torch.zeros(int(L.lh2hip_dn_dw_workspace_bytes(cin, cout)) // 4, device="cuda")
        gw, gb = torch.full((9 * cout * cin,), 7.0, device="cuda"), torch.full((cout,), 7.0, device="cuda")
        assert L.lh2hip_dn_conv3x3_dw(dx.data_ptr(), cin, dgy.data_ptr(), cout, H, W, gw.data_ptr(), gb.data_ptr(), ws.data_ptr(), sh) == 0
        torch.cuda.synchronize()
        check_dw(torch, x, gy, gw, gb, (cin, cout, H, W))


@pytest.mark.parametrize("H,W", [(126, 254), (250, 254), (254, 256)])
def test_light_layers_on_both_sides_of_their_line(torch_cuda, H, W):
    """16 -> 32 and 32 -> 16 take small tiles up to 255 tiles of 64 x 4 (here 128, 252 and 256): equal to crops of 28 x 28, bit for bit."""
    torch = torch_cuda
    L = lh.library()
    sh = torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(H + W)
    x = R.bf16(rng.standard_normal((H, W, 32)))
    w = dev(torch, R.bf16(rng.standard_normal((9, 32, 16)) * 0.2))
    b = torch.from_numpy(rng.standard_normal(32).astype(np.float32)).cuda()

    def run(y0, x0, h, w_):
        cut = x[y0:y0 + h, x0:x0 + w_]
        a16, a32 = dev(torch, np.ascontiguousarray(cut[..., :16])), dev(torch, np.ascontiguousarray(cut))
        o = empty(torch, h * w_ * 32), torch.full((h * w_ * 16,), 7.0, device="cuda")
        assert L.lh2hip_dn_conv3x3(a16.data_ptr(), 16, w.data_ptr(), b.data_ptr(), o[0].data_ptr(), 32, h, w_, 1, sh) == 0
        assert L.lh2hip_dn_conv3x3(a32.data_ptr(), 32, w.data_ptr(), b.data_ptr(), o[1].data_ptr(), 16, h, w_, 2, sh) == 0
        torch.cuda.synchronize()
        return o[0].view(h, w_, 32), o[1].view(h, w_, 16)

    full = run(0, 0, H, W)
    for y0 in (0, H // 2 - 11, H - 28):
        for x0 in (0, W // 2 - 13, W - 28):
            t, l, e, r = (1 if y0 else 0), (1 if x0 else 0), 28 - (y0 + 28 < H), 28 - (x0 + 28 < W)
            for f, p in zip(full, run(y0, x0, 28, 28)):
                assert torch.equal(f[y0 + t:y0 + e, x0 + l:x0 + r], p[t:e, l:r]), (y0, x0)
