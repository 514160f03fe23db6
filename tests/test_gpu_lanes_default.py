"""The default lanes per ray follow the rays marched and the schedule's room; the image does not."""
import pytest

pytestmark = pytest.mark.gpu


# 256 x 128 rays in 16 x 4 tiles: 512; at 2, 4, 8 lanes per ray 1024, 2048, 4096
@pytest.mark.parametrize("room", [512, 1023, 1024, 2048, 4095, 4096])
def test_a_schedule_of_any_room_marches_a_small_frame(mm, gpu, room):
    import torch

    W, H = 256, 128
    ns = mm.NoiseSet("fast")
    ns.generate(mm.noise_params(), mm.current_stream())
    ubos = mm.build_ubos(mm.scenario_scene(aspect=W / H))
    want = torch.zeros(W * H * 4, device="cuda")
    mm.march_clouds(*ubos, ns, want, W, H, params=mm.march_params("scenario", lanes_per_ray=1))
    sched = mm.MarchSchedule(room)
    prm = mm.march_params("scenario")
    for _ in range(3):  # the default order, then longest first
        got = torch.full_like(want, -1.0)
        mm.march_clouds(*ubos, ns, got, W, H, params=prm, schedule=sched)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
    small = mm.MarchSchedule(511)
    with pytest.raises(mm.MMError):
        mm.march_clouds(*ubos, ns, got, W, H, params=prm, schedule=small)


@pytest.mark.parametrize("W,H", [(1, 1), (5, 3), (61, 37), (300, 150), (301, 150)])  # 16 lanes up to 45 000 rays
@pytest.mark.parametrize("preset,over", [
    ("scenario", {}),
    ("scenario", {"max_coarse_steps": 17, "max_fine_steps": 21}),
    ("scenario", {"miss_limit": 1, "opacity_cutoff": 0.3}),
    ("scenario", {"max_steps": 35}),
    ("reference", {"max_steps": 16, "miss_limit": 2}),
    ("reference", {"opacity_cutoff": -1.0}),
])
def test_default_lanes_equal_one_lane(mm, gpu, W, H, preset, over):
    import torch

    ns = mm.NoiseSet("fast", weather_dim=128, low_dim=32, hi_dim=16)
    ns.generate(mm.noise_params(seed=3, weather_seed=5, coverage=0.7), mm.current_stream())
    ubos = mm.build_ubos(mm.scenario_scene(aspect=W / H, pitch_deg=12.0, time=90.0))
    sched = mm.MarchSchedule()
    for phase in (-1, 0):
        got = []
        for lanes, s in ((1, None), (0, None), (0, sched), (0, sched)):
            out = torch.full((W * H * 4,), -1.0, dtype=torch.float32, device="cuda")
            counts = torch.zeros(4, dtype=torch.int64, device="cuda")
            mm.march_clouds(*ubos, ns, out, W, H, phase=phase, params=mm.march_params(preset, lanes_per_ray=lanes, **over),
                            counts=counts, schedule=s)
            torch.cuda.synchronize()
            got.append((out.view(torch.int32), counts.tolist()))
        for o, n in got[1:]:
            assert torch.equal(o, got[0][0]) and n == got[0][1], phase
