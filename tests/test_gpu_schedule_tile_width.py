"""A tile width asked for through a schedule selects the one-lane kernel, which alone has it, whatever the number of
rays: a schedule too small for those tiles refuses the launch, one that holds them marches the same image."""
import numpy as np
import pytest

from test_gpu_schedule import _march, _noise, _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H,width,tiles", [(8, 64, 32, 32), (8, 64, 16, 16), (33, 40, 8, 25), (200, 100, 32, 350)])
def test_tile_width_through_a_schedule(mm, gpu, W, H, width, tiles):
    ns = _noise(mm)
    ubos = _scene(mm, W, H)
    prm = mm.march_params("scenario", tile_width=width)
    ref, cref = _march(mm, ns, ubos, W, H, mm.march_params("scenario"))
    small = mm.MarchSchedule(tiles - 1)
    with pytest.raises(mm.MMError) as e:
        _march(mm, ns, ubos, W, H, prm, schedule=small)
    assert e.value.code == mm.MM_E_SIZE
    small.close()
    sched = mm.MarchSchedule(tiles)
    for _ in range(3):
        got, cgot = _march(mm, ns, ubos, W, H, prm, schedule=sched)
        assert np.array_equal(got, ref)
        assert (cgot == cref).all()
    sched.close()
