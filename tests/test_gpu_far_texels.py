"""Texel coordinates far from the origin. The sampler rounds a coordinate x to 1/256 as floor(256 x + 0.5) with the
addition rounded to float, as the restatement does: from 2^15 texels on (256 x of 2^23 or more) that addition
ties to even, so odd codes move up by one, and the exact floor(256 x + 0.5) would give another weight."""
import numpy as np
import pytest

from test_gpu_march import check_parity, gpu_march, tex, upload  # noqa: F401  (tex is a fixture)
from test_gpu_shadow import _points

pytestmark = pytest.mark.gpu

# Largest texel coordinates in these scenes: inside 2^15, across 2^15 .. 2^16, beyond 2^16.
REACH = [12_000.0, 30_000.0, 60_000.0, 200_000.0]


@pytest.mark.parametrize("fset", ["ref", "fast"])
@pytest.mark.parametrize("reach", REACH)
def test_far_shadow_reads_equal_oracle(mm, gpu, orc, tex, fset, reach):
    import torch

    cam, sun, sky = mm.build_ubos(mm.scenario_scene(aspect=1.0, sun_elevation_deg=40.0, time=0.0))
    ns = upload(mm, tex, fset)
    prm = mm.shadow_params()
    # the points spread over +-20 km, times the march's origin scale of 4: x and z up to 80 km
    prm.low_scale = reach / (128 * 80_000.0)
    prm.weather_scale = reach / (512 * 80_000.0)
    pts = _points(4096, 11)
    out = torch.full((len(pts),), -1.0, dtype=torch.float32, device="cuda")
    mm.cloud_shadow(cam, sun, sky, ns, torch.from_numpy(pts).cuda(), out, params=prm)
    torch.cuda.synchronize()
    ref = orc.cloud_shadow(cam, sun, sky, tex["weather"], tex["low"], pts, prm)
    got = out.cpu().numpy()
    print(fset, reach, "nonzero", float((ref > 0).mean()), "different", int((got != ref).sum()), flush=True)
    assert (ref > 0).mean() > 0.01  # the case exercises clouds
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("lanes", [1, 8])
@pytest.mark.parametrize("reach", REACH)
def test_far_march_reads_match_oracle(mm, gpu, orc, tex, reach, lanes):
    """The same for the march, whose hits lie within some tens of kilometres of the camera."""
    W, H = 96, 64
    cam, sun, sky = mm.build_ubos(mm.scenario_scene(aspect=W / H, sun_elevation_deg=30.0, time=0.0))
    prm = mm.march_params("scenario", lanes_per_ray=lanes)
    for field, n in (("low_scale", 128), ("hi_scale", 32), ("curl_scale", 128)):
        setattr(prm, field, reach / (n * 30_000.0))
    g = gpu_march(mm, upload(mm, tex, "ref"), cam, sun, sky, W, H, params=prm)
    r = orc.march(cam, sun, sky, orc.textures(tex["weather"], tex["curl"], tex["low"], tex["hi"]), prm, W, H)
    assert r[..., 3].min() < 0.9  # the case exercises clouds
    check_parity(g, r, f"reach {reach} lanes {lanes}")
