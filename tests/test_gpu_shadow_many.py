"""Cloud shadows of more points than three 32-bit coordinates' index can count: the last points' values are those of
a call with these points alone."""
import pytest

from test_gpu_march import tex, upload  # noqa: F401  (tex is a fixture)
from test_gpu_shadow import _points

pytestmark = pytest.mark.gpu


def test_points_beyond_a_32_bit_coordinate_index(mm, gpu, tex):
    import torch

    n, tail = (1 << 32) // 3 + 500, 1000  # 3 i wraps for the last 500 of the tail
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs 23 GB of device memory")
    cam, sun, sky = mm.build_ubos(mm.scenario_scene(aspect=1.0, sun_elevation_deg=40.0, time=0.0))
    ns = upload(mm, tex, "fast")
    prm = mm.shadow_params(steps=2)
    last = torch.from_numpy(_points(tail, 3)).cuda()
    want = torch.full((tail,), -1.0, device="cuda")
    mm.cloud_shadow(cam, sun, sky, ns, last, want, params=prm)
    assert (want > 0).sum() > 10  # the case exercises clouds
    points = torch.zeros((n, 3), dtype=torch.float32, device="cuda")
    points[-tail:] = last
    out = torch.full((n,), -1.0, dtype=torch.float32, device="cuda")
    mm.cloud_shadow(cam, sun, sky, ns, points, out, params=prm)
    torch.cuda.synchronize()
    assert torch.equal(out[-tail:], want)
    assert bool((out[:-tail] == out[0]).all())
    del points, out
    torch.cuda.empty_cache()
