"""A schedule shared by launches of the fixed-point and the float sampler. The float sampler's plain march runs on
the lock-step kernel, which takes no schedule: a launch of it between two scheduled ones must leave the record
such that every tile of the next ordered launch is marched once."""
import numpy as np
import pytest

from test_gpu_schedule import _march, _noise, _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("surrogate,lanes", [(False, 0), (False, 1), (False, 2), (False, 8), (True, 0), (True, 1), (True, 2)])
def test_float_launch_between_scheduled_ones(mm, gpu, lanes, surrogate):
    W, H = 640, 400
    ns = _noise(mm)
    over = {}
    if surrogate:
        model = mm.Surrogate(seed=3)
        over = {"cone_mode": mm.CONE_SURROGATE, "surrogate_threshold": 0.0, "surrogate": model.ptr}
    ubos = _scene(mm, W, H)
    prm = {bits: mm.march_params("scenario", lanes_per_ray=lanes, subtexel_bits=bits, **over) for bits in (8, 0)}
    ref = {bits: _march(mm, ns, ubos, W, H, prm[bits]) for bits in (8, 0)}
    sched = mm.MarchSchedule(1 << 16)
    for rep, bits in enumerate([8, 0, 8, 8, 0, 0, 8]):
        got, cgot = _march(mm, ns, ubos, W, H, prm[bits], schedule=sched)
        assert np.array_equal(got, ref[bits][0]), (rep, bits)
        assert (cgot == ref[bits][1]).all(), (rep, bits, cgot, ref[bits][1])
    sched.close()
