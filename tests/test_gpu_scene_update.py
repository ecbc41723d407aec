"""SetGeometry's triangle records, which from 4 MB on (20,165 records) go up beside
the build on a thread of their own, and SetInstance's transforms."""
import numpy as np
import pytest

import lighthouse2_amd as lh
from lighthouse2_amd import scenes
from test_gpu_trace import gpu_closest
from test_oracle import _random_rays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 65, 20164, 20165, 66000])
@pytest.mark.parametrize("refit", [0, 1])
def test_largest_material_of_the_records(torch_cuda, n, refit):
    """A frame is refused exactly while a record's material lies beyond the table,
    wherever that record is and whatever the mesh held before."""
    core = lh.RenderCore()
    core.SetTarget(16, 16, 1)
    core.Setting("refit", refit)
    view = scenes.camera_view((0.0, 0.0, -3.0), (0.0, 0.0, 0.0), 40.0, 16, 16)
    s = scenes.random_triangle_scene(n, seed=n, with_tris=True)
    v, t = s.meshes[0]
    mats = np.concatenate([lh.formats.lambert_material((0.5, 0.4, 0.3))] * 3)
    core.SetMaterials(mats)
    for at in (0, n - 1, n // 2):
        for worst, good in ((3, False), (2, True), (0xffffffff, False), (0, True)):
            t["material"] = 0
            t["material"][at] = worst
            core.SetGeometry(0, v, t)
            core.SetInstance(0, 0)
            core.FinalizeInstances()
            if good:
                core.Render(view, lh.LH2_RESTART)
            else:
                with pytest.raises(lh.LH2HIPError):
                    core.Render(view, lh.LH2_RESTART)
    core.Shutdown()


def test_transforms_of_any_form(torch_cuda):
    T = np.arange(16, dtype=np.float64).reshape(4, 4) * 0.01 + np.eye(4)
    v = scenes.random_triangles(300, 2, sigma=0.1)
    rays = _random_rays(np.random.default_rng(3), 2000)
    got = []
    for form in (T.astype(np.float32), np.asfortranarray(T), T.tolist(), T.reshape(16), np.repeat(T, 2, 1)[:, ::2]):
        core = lh.RenderCore()
        core.SetGeometry(0, v)
        core.SetInstance(0, 0, form)
        core.FinalizeInstances()
        got.append(gpu_closest(torch_cuda, core, rays).view(np.uint32))
        for wrong in (np.eye(3), np.zeros(17), np.zeros((0,))):
            with pytest.raises(ValueError):
                core.SetInstance(0, 0, wrong)
        core.Shutdown()
    assert all(np.array_equal(got[0], g) for g in got[1:])
    assert len(np.unique(got[0])) > 300
