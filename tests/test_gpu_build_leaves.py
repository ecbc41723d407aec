"""The builder with leaves larger than a wave's share (512 primitives): every
primitive in one leaf, boxes of leaves and nodes, and the leaf rules."""
import ctypes

import numpy as np
import pytest

import lighthouse2_amd as lh
from test_trace_stack import LIB

pytestmark = pytest.mark.gpu


def build(torch, lo, hi, max_leaf, max_degenerate):
    lh.library()                                    # the HIP runtime of the process
    check = ctypes.CDLL(LIB).check_build
    check.restype, check.argtypes = ctypes.c_int64, [ctypes.c_void_p] * 2 + [ctypes.c_int] * 3 + [ctypes.c_void_p] * 3 + [ctypes.c_uint64]
    n = len(lo)
    dlo, dhi = (torch.from_numpy(np.ascontiguousarray(np.column_stack([a, np.zeros(n)]).astype(np.float32))).cuda() for a in (lo, hi))
    nodes, prims = torch.full((2 * n, 8), -7, dtype=torch.int32, device="cuda"), torch.full((n,), -7, dtype=torch.int32, device="cuda")
    need = check(None, None, n, 0, 0, None, None, None, 0)
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    count = check(dlo.data_ptr(), dhi.data_ptr(), n, max_leaf, max_degenerate, nodes.data_ptr(), prims.data_ptr(), ws.data_ptr(), need)
    torch.cuda.synchronize()
    assert count > 0
    return nodes[:count].cpu().numpy().view(lh.formats.BuildNode).reshape(-1), prims.cpu().numpy()


@pytest.mark.parametrize("n", [300, 513, 2048, 2049, 5000])
@pytest.mark.parametrize("kind", ["coincident", "cluster", "overlapping"])
def test_large_leaves(torch_cuda, kind, n):
    rng = np.random.default_rng(n)
    c = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    if kind == "coincident":
        c[:] = 0.25
    elif kind == "cluster":
        c[rng.permutation(n)[: n * 2 // 3]] = 0.25
    half = np.float32(0.5) if kind == "overlapping" else np.float32(2.0 ** -6)
    if kind == "overlapping":
        c *= np.float32(1e-5)                       # a split saves at most n * 4e-5 of a box: not worth a node
    lo, hi = c - half, c + half
    nodes, prims = build(torch_cuda, lo, hi, n if kind == "overlapping" else 4, n)
    leaf = nodes["count"] > 0
    assert sorted(prims) == list(range(n))
    first, count = nodes["leftFirst"][leaf], nodes["count"][leaf]
    assert count.sum() == n and len(np.unique(first)) == len(first)
    for x in np.nonzero(leaf)[0]:
        p = prims[nodes["leftFirst"][x]: nodes["leftFirst"][x] + nodes["count"][x]]
        assert np.array_equal(nodes["lo"][x], lo[p].min(0)) and np.array_equal(nodes["hi"][x], hi[p].max(0))
    if kind == "cluster":
        assert count.max() == n * 2 // 3
    else:
        assert len(nodes) == 1
