"""normalize on the device against IEEE float32 in numpy, bit for bit, at the magnitudes where its 1 / sqrt
changes form: squares that are subnormal, around 2^-96, ordinary, and that overflow."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lo,hi", [(-76, -70), (-52, -44), (-2, 2), (60, 66)])
def test_normalize_magnitudes(ctx, lo, hi):
    rng = np.random.default_rng(hi - lo)
    mid = np.float32([[0.5, 0.5]])   # the centre ray: the direction is normalize(znear * forward)
    z = np.exp2(rng.uniform(lo, hi, 48)).astype(np.float32)
    z = np.concatenate([z, np.exp2(np.arange(lo, hi + 1)).astype(np.float32)])
    got = np.float32([ctx.diag_camera(np.float32([0, 0, 0, 0, 0, -1, 0, 1, 0, v, 1e30, 0.7, 1.0]), mid)[0, 6] for v in z])
    with np.errstate(over="ignore", under="ignore", divide="ignore"):
        s = z * z
        ref = np.where(s > 0, -z * (np.float32(1) / np.sqrt(s)), -z)
    assert ref.dtype == np.float32
    np.testing.assert_array_equal(got, ref)
