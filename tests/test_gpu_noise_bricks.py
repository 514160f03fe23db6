"""Generator sizes at the edges of the kernels' blocks, against the oracle byte for byte: curl maps whose texels
do not fill a block of 64, and volumes smaller than a brick of 8 x 8 x 4, with partial bricks and of whole ones."""
import pytest

import fmt_util as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("curl,low,hi", [(7, 4, 3), (8, 8, 8), (65, 9, 33), (100, 72, 40)])
def test_small_and_partial_blocks(mm, gpu, orc, curl, low, hi):
    import torch

    orc.L.orc_set_curl_mutation(0)
    ns = mm.NoiseSet("ref", curl_dim=curl, low_dim=low, hi_dim=hi)
    ns.generate(mm.noise_params(seed=19, what=mm.GEN_CURL | mm.GEN_LOW_RES | mm.GEN_HI_RES), mm.current_stream())
    torch.cuda.synchronize()
    assert ns.curl.tensor.cpu().numpy().tobytes() == orc.curl(curl)[0].tobytes()
    assert ns.low_res.tensor.cpu().numpy().tobytes() == F.pack_low(orc.low_res(low, 19), F.FMT_RGBA8, F.LAYOUT_LINEAR)
    assert ns.hi_res.tensor.cpu().numpy().tobytes() == F.pack_hi(orc.hi_res(hi, 19), F.FMT_RGBA8, F.LAYOUT_LINEAR)


@pytest.mark.parametrize("dim", [1, 5, 16, 17, 33, 100, 257])  # one texel, partial tiles, lattices finer than texels
@pytest.mark.parametrize("fset", ["ref", "fast"])
def test_weather_sizes(mm, gpu, orc, dim, fset):
    import torch

    ns = mm.NoiseSet(fset, weather_dim=dim)
    ns.generate(mm.noise_params(weather_seed=23, coverage=0.6, what=mm.GEN_WEATHER), mm.current_stream())
    torch.cuda.synchronize()
    want = orc.weather(dim, 23, 0.6)
    fmt, layout = (F.FMT_RGBA8, F.LAYOUT_LINEAR) if fset == "ref" else (F.FMT_RG8, F.LAYOUT_APRON)
    assert ns.weather.tensor.cpu().numpy().tobytes() == F.pack_weather(want, fmt, layout)
