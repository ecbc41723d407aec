"""The short forms of division, reciprocal, square root, exponential and the bf16
conversion against correctly rounded ones, bit for bit: images and gradients are
defined by these bits."""
import ctypes

import numpy as np
import pytest

import lighthouse2_amd as lh
from test_trace_stack import LIB

pytestmark = pytest.mark.gpu
RCP, SQRT, DIV, EXP_NEG, EXP = range(5)


def short(torch, which, a, b=None):
    lh.library()                                    # the HIP runtime of the process
    check = ctypes.CDLL(LIB).check_short
    check.argtypes = [ctypes.c_int] + [ctypes.c_void_p] * 3 + [ctypes.c_int]
    out = torch.zeros_like(a)
    torch.cuda.synchronize()
    assert check(which, a.data_ptr(), None if b is None else b.data_ptr(), out.data_ptr(), a.numel()) == 0
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("exponent", [-100, -99, -51, -2, -1, 0, 1, 2, 50, 98, 99])
def test_reciprocal_and_square_root(torch_cuda, exponent):
    """Every float of binades at the ends and in the middle of [2^-100, 2^100); an estimate depends on the mantissa and,
    for the square root, on whether the exponent is odd."""
    bits = torch_cuda.arange(1 << 23, dtype=torch_cuda.int32, device="cuda") | ((exponent + 127) << 23)
    x = bits.view(torch_cuda.float32)
    h = x.cpu().numpy()
    assert np.array_equal(short(torch_cuda, RCP, x).cpu().numpy().view(np.uint32), (np.float32(1) / h).view(np.uint32))
    assert np.array_equal(short(torch_cuda, SQRT, x).cpu().numpy().view(np.uint32), np.sqrt(h).view(np.uint32))


def test_division(torch_cuda):
    """Random pairs of the denoiser's range: denominators of [1e-5, 1e30], quotients that neither overflow nor are denormal."""
    rng = np.random.default_rng(1)
    n = 1 << 24
    num = (10.0 ** rng.uniform(-20, 30, n)).astype(np.float32)
    den = (10.0 ** rng.uniform(-5, 30, n)).astype(np.float32)
    num[: n // 2] = den[: n // 2] * (10.0 ** rng.uniform(-3, 3, n // 2)).astype(np.float32)     # and near one another, as depths are
    num[:3], den[:3] = (0.0, 1.0, 3.0), (1e-5, 1.0, 3.0)
    den = np.clip(den, np.float32(1e-5), np.float32(1e30))
    with np.errstate(over="ignore"):
        want = num / den
    ok = np.isfinite(want) & np.isfinite(num) & ((want >= 1.2e-38) | (num == 0)) & ((num >= 1e-20) | (num == 0))
    got = short(torch_cuda, DIV, *(torch_cuda.from_numpy(a).cuda() for a in (num, den))).cpu().numpy()
    assert ok.sum() > n // 2
    assert np.array_equal(got[ok].view(np.uint32), want[ok].view(np.uint32))


def test_exponential_of_negative_numbers(torch_cuda):
    """Every float from -0 to -infinity, and NaN."""
    for k in range(8):
        x = (torch_cuda.arange(1 << 28, dtype=torch_cuda.int32, device="cuda") + (k - 8) * (1 << 28)).view(torch_cuda.float32)
        a, b = short(torch_cuda, EXP_NEG, x), short(torch_cuda, EXP, x)
        nan = torch_cuda.isnan(x)
        assert torch_cuda.equal(torch_cuda.isnan(a), nan) and torch_cuda.equal(torch_cuda.isnan(b), nan)
        assert bool(((a.view(torch_cuda.int32) == b.view(torch_cuda.int32)) | nan).all()), k


def test_bf16_conversion(torch_cuda):
    """Every float, through the Adam step's bf16 copy: round to nearest even, NaN quiet with its upper bits."""
    torch = torch_cuda
    sh = torch.cuda.current_stream().cuda_stream
    n = 1 << 27
    out = torch.zeros(n, dtype=torch.int16, device="cuda")
    for k in range(32):
        u = torch.arange(n, dtype=torch.int32, device="cuda") + (k - 16) * n
        assert lh.library().lh2hip_dn_adam(u.data_ptr(), u.data_ptr(), u.data_ptr(), None, n, 0.0, 0.9, 0.999, 1e-8, 1, out.data_ptr(), None, 0, 0, sh) == 0
        w = u.to(torch.int64) & 0xffffffff
        want = torch.where((w & 0x7fffffff) > 0x7f800000, (w >> 16) | 0x40, (w + 0x7fff + ((w >> 16) & 1)) >> 16) & 0xffff
        assert torch.equal(out.to(torch.int64) & 0xffff, want), k
