"""The lanes that share a shaded point's steps: any number of points and steps gives the values of one lane
per point, also for points out of every range."""
import numpy as np
import pytest

from test_gpu_march import tex, upload  # noqa: F401  (tex is a fixture)
from test_gpu_shadow import _points

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [0, 1, 2, 5, 6, 9, 40])
def test_split_steps_equal_one_lane(mm, gpu, tex, steps):
    import torch

    cam, sun, sky = mm.build_ubos(mm.scenario_scene(aspect=1.0, sun_elevation_deg=12.0, time=300.0))
    ns = upload(mm, tex, "fast")
    prm = mm.shadow_params()
    prm.steps = steps
    pts = _points(65537, 9)  # one lane per point above 65536 points
    pts[5], pts[6], pts[7] = np.inf, np.nan, -3e38
    pts = torch.from_numpy(pts).cuda()

    def run(n):
        out = torch.full((n,), -1.0, dtype=torch.float32, device="cuda")
        mm.cloud_shadow(cam, sun, sky, ns, pts[:n].contiguous(), out, params=prm)
        torch.cuda.synchronize()
        return out.view(torch.int32)

    whole = run(65537)
    for n in (1, 9, 32768, 32769, 65536):
        assert torch.equal(run(n), whole[:n]), n
