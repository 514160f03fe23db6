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
