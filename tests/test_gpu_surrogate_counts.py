"""Counting launches of the surrogate-lit march: the same image as without counters, for both texture sets, both
step rules, both samplers and either number of lanes per ray, with every light cone marched (threshold 0, where
the image is the plain march's) and with none."""
import numpy as np
import pytest

from test_gpu_march import gpu_march, tex, upload  # noqa: F401  (tex is a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fset", ["ref", "fast"])
@pytest.mark.parametrize("preset", ["scenario", "reference"])
@pytest.mark.parametrize("bits", [8, 0])
def test_counted_surrogate_march_equals_uncounted(mm, gpu, tex, fset, preset, bits):
    W, H = 203, 117  # ragged tiles: batches of every size
    ubos = mm.build_ubos(mm.scenario_scene(aspect=W / H, sun_elevation_deg=20.0, time=60.0))
    ns = upload(mm, tex, fset)
    model = mm.Surrogate(seed=3)
    plain = gpu_march(mm, ns, *ubos, W, H, params=mm.march_params(preset, subtexel_bits=bits))
    seen = {}
    for threshold in (0.0, 1e30):
        for lanes in (1, 2):
            prm = mm.march_params(preset, subtexel_bits=bits, lanes_per_ray=lanes, cone_mode=mm.CONE_SURROGATE,
                                  surrogate_threshold=threshold, surrogate=model.ptr)
            image = gpu_march(mm, ns, *ubos, W, H, params=prm)
            counted, counts = gpu_march(mm, ns, *ubos, W, H, params=prm, counts=True)
            assert np.array_equal(counted, image), (threshold, lanes)
            if threshold == 0.0:
                assert np.array_equal(counted, plain), lanes
                assert counts[2] == counts[3] > 0  # every cone is marched
            else:
                assert counts[3] == 0 and counts[2] > 0
            seen.setdefault(threshold, []).append((image, counts))
    for (a, ca), (b, cb) in seen.values():
        assert np.array_equal(a, b) and (ca == cb).all()
