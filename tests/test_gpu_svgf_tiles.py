"""The staged a-trous passes and the branch-free history reads against the
oracle, bit for bit: image sizes at the edges of a pass's lattices (16 x 16
pixels 1, 2 and 4 apart), and depths and depth derivatives from misses and
grazing planes: huge, infinite, and beyond the range of the short division."""
import numpy as np
import pytest

import lighthouse2_amd as lh
from lighthouse2_amd import scenes
import oracle as orc
from lighthouse2_amd.scenes import gbuffer

pytestmark = pytest.mark.gpu


def run(torch, w, h, wild, frames=2):
    rng = np.random.default_rng(w * 1000 + h)
    g, o = lh.Svgf(w, h, taa=True), orc.OracleSvgf(w, h)
    out = torch.zeros((h, w, 4), dtype=torch.float32, device="cuda")
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    view = scenes.camera_view((0.5, 0.6, -1.0), (0.5, 0.5, 1.0), 50.0, w, h)
    for k in range(frames):
        acc, feat, wp, dd = gbuffer(view, w, h, seed=3 + k, spec_strip=w > 8)
        if wild:
            m = rng.random((h, w))
            feat[..., 2][m < 0.2] = np.float32(1e34).view(np.uint32)        # misses
            dd[m < 0.2] = 0
            for lo, hi, value in ((0.2, 0.3, 1e12), (0.3, 0.4, -3e29), (0.4, 0.45, 1e31), (0.45, 0.5, np.inf), (0.5, 0.55, 1e38), (0.55, 0.6, 1e-30)):
                pick = (m >= lo) & (m < hi)
                dd[..., 2][pick], dd[..., 3][pick] = value, -value
            feat[..., 1][m > 0.95] = 0xfffffffc                              # normals longer than 1: weights overflow
        a, f, p, d = dev(acc), dev(feat.view(np.int32)), dev(wp), dev(dd)
        g.frame(a.data_ptr(), f.data_ptr(), p.data_ptr(), d.data_ptr(), view, out.data_ptr(), j=(0.1, 0.0))
        torch.cuda.synchronize()
        ref = o.frame(acc, feat, wp, dd, view, j=(0.1, 0.0), samples=1, taa=True)
        assert np.array_equal(out.cpu().numpy()[1:-1, 1:-1].view(np.uint32), ref[1:-1, 1:-1].view(np.uint32)), (w, h, k)
        for which in range(7):
            assert np.array_equal(g.read(which).view(np.uint32), o.read(which).view(np.uint32)), (w, h, k, which)
    g.close()


@pytest.mark.parametrize("w,h", [(3, 3), (4, 17), (16, 16), (17, 15), (33, 31), (63, 65), (64, 64), (65, 63), (130, 70)])
def test_lattice_edges(torch_cuda, w, h):
    run(torch_cuda, w, h, False)


@pytest.mark.parametrize("w,h", [(40, 24), (97, 50)])
def test_wild_depths(torch_cuda, w, h):
    run(torch_cuda, w, h, True)
