"""Post chain where its kernels change paths: images of more than a million pixels (four rows a lane) with rows
of taps farther apart than the rows are or in reverse order, images of one to a few texels and of one block more, taps that
leave the image, weights coarser than 1/256, sample counts around a batch of four, a sun on a pixel centre (no
direction to blur along) or far outside, and image values that are not ordinary numbers -- bit for bit."""
import numpy as np
import pytest

from test_gpu_post import _run
from test_oracle_post import _ubos

pytestmark = pytest.mark.gpu


def _same(a, b):
    return np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)].view(np.uint32),
                                                                      b[~np.isnan(b)].view(np.uint32))


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("W,H,pitch,bits,samples,sun,density", [
    (1, 1, 1, 8, 8, (0.3, 0.2), 0.5),
    (2, 1, 3, 8, 4, (0.3, 0.2), 0.5),
    (1, 40, 2, 8, 5, (0.1, -0.4), 0.5),
    (17, 2, 17, 8, 1, (0.0, 0.0), 0.5),
    (65, 33, 80, 8, 9, (2.0 * 20.5 / 65 - 1.0, 2.0 * 9.5 / 33 - 1.0), 0.5),
    (96, 64, 96, 8, 8, (0.0, 0.99), 0.5),
    (129, 67, 129, 7, 6, (-0.2, 0.1), 0.5),
    (128, 72, 128, 8, 11, (-400.0, 3.0), 0.5),
    (128, 72, 128, 8, 7, (3e37, 1e30), 0.5),
    (128, 72, 128, 8, 6, (0.1, 0.2), 1.7),
    (1027, 1025, 1031, 8, 8, (0.3, 0.2), 0.5),
    (1027, 1025, 1031, 8, 5, (0.1, -0.1), 1.9),
    (1026, 1023, 1026, 8, 6, (-0.2, 0.95), -0.4),
])
def test_edges_match_the_oracle(mm, gpu, orc, W, H, pitch, bits, samples, sun, density, special):
    rng = np.random.default_rng(W + H)
    img = rng.uniform(0.0, 2.0, (H, W, 4)).astype(np.float32)
    if special:
        odd = np.array([0.0, -0.0, 1e-40, -1.0, np.inf, -np.inf, np.nan, 3e38, 1e9, 1.1e9, 1e-30], np.float32)
        at = rng.random((H, W, 4)) < 0.03
        img[at] = rng.choice(odd, int(at.sum()))
    cam, s = _ubos(mm, sx=sun[0], sy=sun[1])
    p = mm.post_params(subtexel_bits=bits, god_ray_samples=samples, god_ray_density=density)
    with np.errstate(all="ignore"):
        oa, oh, oo = orc.post_process(cam, s, img, p)
    ga, gh, go = _run(mm, cam, s, img, p, pitch)
    assert _same(ga, oa) and _same(gh, oh) and np.array_equal(go, oo)
