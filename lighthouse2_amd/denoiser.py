"""Learned denoiser: a 5-level convolutional U-Net (3x3 kernels, 32 channels)
trained and run with the gfx950 kernels of librendercore_hip.so (bf16 NHWC
activations and weights, fp32 accumulation on the matrix cores). No
counterpart in the reference, whose denoisers are SVGF and OptiX's.

Network (channels): input 16 = [radiance 3, albedo 3, normal 3, depth 1, 0 x 6]
  encoder level l = 0..3: a = relu(conv(in)), b = relu(conv(a)), in_{l+1} = avgpool2(b)
  bottleneck (level 4):   a = relu(conv(in)), b = relu(conv(a))
  decoder level l = 3..0: cat = [upsample2(prev), b_l], c = relu(conv(cat)), d = relu(conv(c))
                          (read from its two halves, forward and backward: never materialised)
  output: conv(d_0) -> 16 channels fp32, the first 3 are the denoised radiance.
Loss: relMSE over the 3 output channels. Optimiser: Adam on fp32 master weights.
Torch tensors serve as device buffers only; every operation is a kernel of
the library (lh2hip_dn_*).
"""
import ctypes
import struct

import numpy as np

from .core import library, _check

LEVELS = 5
CH = 32
CIN = 16
COUT = 16


class _Layer(ctypes.Structure):
    """lh2hip_dn_layer: one convolution's weight gradient."""
    _fields_ = [(n, ctypes.c_void_p) for n in ("x", "coarse", "dy", "dw", "db")] + [(n, ctypes.c_int) for n in ("Cin", "Cout", "H", "W")]


class _Tensor(ctypes.Structure):
    """lh2hip_dn_tensor: one parameter tensor of an Adam step."""
    _fields_ = ([(n, ctypes.c_void_p) for n in ("p", "m", "v", "g", "wfwd", "wbwd")] + [("n", ctypes.c_uint64)]
                + [(n, ctypes.c_int) for n in ("Cout", "Cin")])


def _records(cls, fields, flat, n):
    """n records from their fields in one go (5 us for 38 tensors; 31 record by record)."""
    return (cls * n).from_buffer_copy(struct.pack(fields * n, *flat)), n


def layer_specs():
    """(name, Cin, Cout) of the 19 convolutions, in forward order."""
    spec = []
    for lvl in range(LEVELS):
        spec.append((f"e1_{lvl}", CIN if lvl == 0 else CH, CH))
        spec.append((f"e2_{lvl}", CH, CH))
    for lvl in range(LEVELS - 2, -1, -1):
        spec.append((f"d1_{lvl}", 2 * CH, CH))
        spec.append((f"d2_{lvl}", CH, CH))
    spec.append(("out", CH, COUT))
    return spec


_SPECS = layer_specs()
# level, input activation and output gradient of each (the decoder's first convolutions read _below their level as well)
_TENSORS = [(int(n[-1]), {"e1": "in", "e2": "a", "d1": "b", "d2": "c"}[n[:2]] + n[2:], {"e1": "a", "e2": "b", "d1": "c", "d2": "d"}[n[:2]] + n[2:])
            for n, _, _ in _SPECS[:-1]] + [(0, "d_0", None)]


def init_params(seed=0):
    """He-normal weights [9][Cout][Cin] and zero biases (float32, numpy)."""
    rng = np.random.default_rng(seed)
    out = {}
    for name, ci, co in layer_specs():
        w = rng.standard_normal((9, co, ci)) * np.sqrt(2.0 / (9 * ci))
        if name == "e1_0":
            w[:, :, 10:] = 0.0                    # padding channels of the input
        if name == "out":
            w[:, 3:, :] = 0.0                     # only 3 output channels are used
        out[name] = (w.astype(np.float32), np.zeros(co, np.float32))
    return out


class UNetDenoiser:
    def __init__(self, H, W, seed=0, params=None, device="cuda"):
        import torch
        if H % 16 or W % 16:
            raise ValueError("image size must be a multiple of 16 (4 pooling steps)")
        self.torch, self.H, self.W = torch, H, W
        self.stream = torch.cuda.current_stream()
        self.sh = self.stream.cuda_stream
        self.t = 0
        bf = dict(dtype=torch.int16, device=device)
        f32 = dict(dtype=torch.float32, device=device)
        self.p = {}
        params = params or init_params(seed)
        for name, ci, co in layer_specs():
            w, b = params[name]
            d = {"ci": ci, "co": co,
                 "w": torch.from_numpy(np.ascontiguousarray(w)).to(device), "b": torch.from_numpy(np.ascontiguousarray(b)).to(device)}
            for k in ("w", "b"):
                d["m" + k] = torch.zeros_like(d[k])
                d["v" + k] = torch.zeros_like(d[k])
                d["g" + k] = torch.zeros_like(d[k])
            d["wf"] = torch.zeros(9 * co * ci, **bf)
            d["wb"] = torch.zeros(9 * co * ci, **bf)
            self.p[name] = d
        self._cast()
        # activations per level (kept for the backward pass) and the gradients of
        # what each layer adds up before its ReLU (kept for the weight gradients)
        self.a, self.g = {}, {}
        for lvl in range(LEVELS):
            h, w = H >> lvl, W >> lvl
            self.a[f"in_{lvl}"] = torch.zeros(h * w * (CIN if lvl == 0 else CH), **bf)
            if lvl > 0:
                self.g[f"in_{lvl}"] = torch.zeros(h * w * CH, **bf)
            for k in ("a", "b") + (("c", "d") if lvl < LEVELS - 1 else ()):
                self.a[f"{k}_{lvl}"] = torch.zeros(h * w * CH, **bf)
                self.g[f"{k}_{lvl}"] = torch.zeros(h * w * CH, **bf)
            if lvl < LEVELS - 1:
                self.g[f"skip_{lvl}"] = torch.zeros(h * w * CH, **bf)
        self.out = torch.zeros(H * W * COUT, **f32)
        self.dout = torch.zeros(H * W * COUT, **bf)
        self.loss = torch.zeros(1, **f32)
        need = int(library().lh2hip_dn_dw_batch_workspace_bytes(*self._layer_table()))
        self.ws = torch.zeros(need // 4, **f32)    # empty (and the backward pass refused) beyond the weight gradient's sizes

    # ---- helpers --------------------------------------------------------
    # Both tables are made for each call: a program may have put other tensors into p, a or g since the last one.
    def _tensor_table(self, grads):
        """Every weight and bias for one Adam launch, and their number; without gradients: the weights' bf16 copies only."""
        flat = []
        for d in self.p.values():
            w = d["w"]
            flat += (w.data_ptr(), d["mw"].data_ptr(), d["vw"].data_ptr(), d["gw"].data_ptr() if grads else 0, d["wf"].data_ptr(),
                     d["wb"].data_ptr(), w.numel(), d["co"], d["ci"])
            if grads:
                b = d["b"]
                flat += (b.data_ptr(), d["mb"].data_ptr(), d["vb"].data_ptr(), d["gb"].data_ptr(), 0, 0, b.numel(), 0, 0)
        return _records(_Tensor, "7Q2i", flat, len(flat) // 9)

    def _layer_table(self):
        """Inputs and output gradients of the 19 convolutions for one weight-gradient launch, and their number."""
        a, g, flat = self.a, self.g, []
        for (name, ci, co), (lvl, x, gy) in zip(_SPECS, _TENSORS):
            d = self.p[name]
            flat += (a[x].data_ptr(), self._below(lvl).data_ptr() if ci == 2 * CH else 0, g[gy].data_ptr() if gy else self.dout.data_ptr(),
                     d["gw"].data_ptr(), d["gb"].data_ptr(), ci, co, self.H >> lvl, self.W >> lvl)
        return _records(_Layer, "5Q4i", flat, len(_SPECS))

    def _below(self, lvl, grad=False):
        """The tensor a decoder level upsamples (or its gradient)."""
        t = self.g if grad else self.a
        return t[f"d_{lvl + 1}"] if lvl + 1 < LEVELS - 1 else t[f"b_{LEVELS - 1}"]

    def _cast(self):
        _check(library().lh2hip_dn_adam_batch(*self._tensor_table(grads=False), 0.0, 0.9, 0.999, 1e-8, 1, self.sh))

    def _conv(self, x, name, y, h, w, flags):
        d = self.p[name]
        _check(library().lh2hip_dn_conv3x3(x.data_ptr(), d["ci"], d["wf"].data_ptr(), d["b"].data_ptr(), y.data_ptr(), d["co"],
                                           h, w, flags, self.sh))

    def _dx_relu(self, gy, name, act, gx, h, w):
        """Gradient of a layer's input, through the ReLU that made the input."""
        d = self.p[name]
        _check(library().lh2hip_dn_conv3x3_dx_relu(gy.data_ptr(), d["co"], d["wb"].data_ptr(), act.data_ptr(), gx.data_ptr(), d["ci"],
                                                   h, w, self.sh))

    # ---- public API -----------------------------------------------------
    def set_input(self, radiance, albedo, normal, depth):
        """Device float32 tensors (H, W, 4) x 3 and (H, W)."""
        _check(library().lh2hip_dn_pack_input(radiance.data_ptr(), albedo.data_ptr(), normal.data_ptr(), depth.data_ptr(),
                                              self.H, self.W, self.a["in_0"].data_ptr(), self.sh))

    def set_input_packed(self, packed_bf16):
        self.a["in_0"].copy_(packed_bf16.reshape(-1))

    def forward(self):
        """Runs the network on the current input; returns the fp32 output (H, W, 16)."""
        self._conv(self.a["in_0"], "e1_0", self.a["a_0"], self.H, self.W, 1)
        self._forward_from_a0()
        self._conv(self.a["d_0"], "out", self.out, self.H, self.W, 2)
        return self.out.view(self.H, self.W, COUT)

    def _forward_from_a0(self):
        """Every layer after e1_0 and before the output convolution."""
        L = library()
        H, W = self.H, self.W
        for lvl in range(LEVELS):
            h, w = H >> lvl, W >> lvl
            if lvl > 0:
                self._conv(self.a[f"in_{lvl}"], f"e1_{lvl}", self.a[f"a_{lvl}"], h, w, 1)
            if lvl < LEVELS - 1:                   # b_l and its 2x2 average in_{l+1} from one kernel
                d = self.p[f"e2_{lvl}"]
                _check(L.lh2hip_dn_conv3x3_pool(self.a[f"a_{lvl}"].data_ptr(), CH, d["wf"].data_ptr(), d["b"].data_ptr(),
                                                self.a[f"b_{lvl}"].data_ptr(), CH, h, w, self.a[f"in_{lvl + 1}"].data_ptr(), self.sh))
            else:
                self._conv(self.a[f"a_{lvl}"], f"e2_{lvl}", self.a[f"b_{lvl}"], h, w, 1)
        prev = self.a[f"b_{LEVELS - 1}"]
        for lvl in range(LEVELS - 2, -1, -1):
            h, w = H >> lvl, W >> lvl
            d = self.p[f"d1_{lvl}"]
            _check(L.lh2hip_dn_conv3x3_cat(prev.data_ptr(), self.a[f"b_{lvl}"].data_ptr(), d["wf"].data_ptr(), d["b"].data_ptr(),
                                           self.a[f"c_{lvl}"].data_ptr(), CH, h, w, 1, self.sh))
            self._conv(self.a[f"c_{lvl}"], f"d2_{lvl}", self.a[f"d_{lvl}"], h, w, 1)
            prev = self.a[f"d_{lvl}"]

    def loss_backward(self, target):
        """relMSE against target (device float32 (H, W, 4)); fills every
        parameter gradient. Returns the loss as a device scalar."""
        L = library()
        H, W = self.H, self.W
        self.loss.zero_()
        _check(L.lh2hip_dn_relmse(self.out.data_ptr(), COUT, target.data_ptr(), H, W, self.dout.data_ptr(), self.loss.data_ptr(), self.sh))
        g, a = self.g, self.a
        self._dx_relu(self.dout, "out", a["d_0"], g["d_0"], H, W)
        for lvl in range(0, LEVELS - 1):
            h, w = H >> lvl, W >> lvl
            self._dx_relu(g[f"d_{lvl}"], f"d2_{lvl}", a[f"c_{lvl}"], g[f"c_{lvl}"], h, w)
            _check(L.lh2hip_dn_conv3x3_dx_cat(g[f"c_{lvl}"].data_ptr(), self.p[f"d1_{lvl}"]["wb"].data_ptr(), self._below(lvl).data_ptr(),
                                              self._below(lvl, grad=True).data_ptr(), g[f"skip_{lvl}"].data_ptr(), h, w, self.sh))
        for lvl in range(LEVELS - 1, -1, -1):
            h, w = H >> lvl, W >> lvl
            if lvl < LEVELS - 1:
                _check(L.lh2hip_dn_pool2_bwd_relu(g[f"in_{lvl + 1}"].data_ptr(), g[f"skip_{lvl}"].data_ptr(), a[f"b_{lvl}"].data_ptr(), CH, h, w,
                                                  g[f"b_{lvl}"].data_ptr(), self.sh))
            self._dx_relu(g[f"b_{lvl}"], f"e2_{lvl}", a[f"a_{lvl}"], g[f"a_{lvl}"], h, w)
            if lvl > 0:
                d = self.p[f"e1_{lvl}"]
                _check(L.lh2hip_dn_conv3x3(g[f"a_{lvl}"].data_ptr(), CH, d["wb"].data_ptr(), None, g[f"in_{lvl}"].data_ptr(), CH, h, w, 0, self.sh))
        _check(L.lh2hip_dn_conv3x3_dw_batch(*self._layer_table(), self.ws.data_ptr(), self.ws.numel() * 4, self.sh))
        return self.loss

    def step(self, lr=1e-3, b1=0.9, b2=0.999, eps=1e-8):
        """One Adam step on every parameter (also refreshes the bf16 copies)."""
        self.t += 1
        _check(library().lh2hip_dn_adam_batch(*self._tensor_table(grads=True), lr, b1, b2, eps, self.t, self.sh))

    def weights_blob(self):
        """The network's inference weights as one blob (the job server's
        lh2hip_server_set_denoiser layout): per layer in forward order, the
        bf16 forward weights [9][Cout][Cin] then the fp32 bias [Cout]."""
        self.torch.cuda.synchronize()
        parts = []
        for name, ci, co in layer_specs():
            d = self.p[name]
            parts.append(d["wf"].cpu().numpy().astype(np.int16).tobytes())
            parts.append(d["b"].cpu().numpy().astype(np.float32).tobytes())
        blob = b"".join(parts)
        assert len(blob) == library().lh2hip_dn_weights_bytes()
        return blob

    def set_input_frame(self, acc32, features, spp, w, h):
        """Input from a filter-estimator frame on the device (acc32 float4
        [2 h w], features uint4 [h w]; the frame's w x h inside this network's
        H x W): the same kernel the job server runs."""
        _check(library().lh2hip_dn_frame_input(acc32.data_ptr(), features.data_ptr(), 1.0 / spp, w, h, self.H, self.W,
                                               self.a["in_0"].data_ptr(), self.sh))

    def denoise_frame(self, acc32, features, spp, w, h, image):
        """Inference on a filter-estimator frame, the output convolution writing
        the display image itself (no fp32 output tensor): the image equals
        set_input_frame + forward + output_frame's."""
        L, H, W = library(), self.H, self.W
        self.set_input_frame(acc32, features, spp, w, h)
        self._conv(self.a["in_0"], "e1_0", self.a["a_0"], H, W, 1)
        self._forward_from_a0()
        d = self.p["out"]
        _check(L.lh2hip_dn_conv3x3_display(self.a["d_0"].data_ptr(), d["wf"].data_ptr(), d["b"].data_ptr(), features.data_ptr(), w, h,
                                           image.data_ptr(), H, W, self.sh))

    def output_frame(self, features, w, h, image):
        """Display image (w x h float4, device) from the last forward pass, as the job server writes it."""
        _check(library().lh2hip_dn_frame_output(self.out.data_ptr(), self.H, self.W, features.data_ptr(), w, h, image.data_ptr(), self.sh))

    def params_numpy(self):
        return {k: (d["w"].cpu().numpy(), d["b"].cpu().numpy()) for k, d in self.p.items()}

    def grads_numpy(self):
        return {k: (d["gw"].cpu().numpy(), d["gb"].cpu().numpy()) for k, d in self.p.items()}

    def flops_forward(self):
        """Multiply-add FLOPs of one forward pass (2 per MAC)."""
        f = 0
        for name, ci, co in layer_specs():
            lvl = 0 if name == "out" else int(name.split("_")[1])
            f += 2 * 9 * ci * co * (self.H >> lvl) * (self.W >> lvl)
        return f


def bf16_bits(a):
    """float32 numpy -> bf16 bits (round to nearest even), as int16."""
    u = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    r = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)
    return r.view(np.int16)


def bf16_to_f32(bits):
    return (np.asarray(bits).astype(np.uint16).astype(np.uint32) << 16).view(np.float32)
