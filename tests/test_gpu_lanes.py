"""The ray-parallel march's round commit at the limits of the loop: image and work counters equal the
one-lane march's for step budgets, counted-step limits, miss limits and opacity cut-offs that end rounds at
every position, in bounded and general stepping."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes", [2, 4, 8])
@pytest.mark.parametrize("preset,over", [
    ("scenario", {"max_coarse_steps": 0}),
    ("scenario", {"max_coarse_steps": 5, "max_fine_steps": 9}),
    ("scenario", {"miss_limit": 1}),
    ("scenario", {"miss_limit": 3, "fine_step_mul": 1.0}),
    ("scenario", {"opacity_cutoff": 0.3}),
    ("scenario", {"max_steps": 7}),
    ("reference", {"max_steps": 1}),
    ("reference", {"max_steps": 13, "miss_limit": 2}),
    ("reference", {"max_coarse_steps": 6, "max_fine_steps": 3}),
    ("reference", {"opacity_cutoff": -1.0}),
])
def test_round_commits_equal_the_loop(mm, gpu, lanes, preset, over):
    import torch

    W, H = 61, 37  # ragged tiles in both axes for every lane count
    ns = mm.NoiseSet("fast", weather_dim=128, low_dim=32, hi_dim=16)
    ns.generate(mm.noise_params(seed=3, weather_seed=5, coverage=0.7), mm.current_stream())
    cam, sun, sky = mm.build_ubos(mm.scenario_scene(aspect=W / H, pitch_deg=12.0, time=90.0))
    got = {}
    for n in (1, lanes):
        out = torch.full((W * H * 4,), -7.0, dtype=torch.float32, device=gpu)
        counts = torch.zeros(4, dtype=torch.int64, device=gpu)
        prm = mm.march_params(preset, lanes_per_ray=n, **over)
        mm.march_clouds(cam, sun, sky, ns, out, W, H, params=prm, counts=counts)
        torch.cuda.synchronize()
        got[n] = (out.cpu(), counts.tolist())
    assert torch.equal(got[1][0].view(torch.int32), got[lanes][0].view(torch.int32))
    assert got[1][1] == got[lanes][1]
