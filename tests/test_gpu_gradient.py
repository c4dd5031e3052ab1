"""Normals of a device field (k_build's gradients): bricks clear of the faces and
the others, volumes written through the caches and past them, and gradients of
every size, against the float32 formula in numpy.

Tolerance: sums, products and quotients are correctly rounded on both sides and
the device's square root is within one ulp, so the norms differ by at most two
ulps (2^-22) after 1e-8 is added and the quotients by one more (2^-23):
2^-21.4 = 3.6e-7 of the value; below the normal numbers, one unit (2^-149)."""

import numpy as np
import pytest

from test_build import _Context

pytestmark = pytest.mark.gpu


def _field(kind, shape):
    rng = np.random.default_rng(sum(shape))
    u = rng.uniform(0.0, 1.0, shape).astype(np.float32)
    if kind == "unit":
        return u
    if kind == "steps":            # zero gradients of either sign, equal neighbours
        return np.where(u < 0.5, -np.float32(0.0), (np.floor(u * 4) / 4).astype(np.float32))
    sign = np.where(u < 0.5, np.float32(-1), np.float32(1))     # both sides of the shared reciprocal's range
    return sign * np.exp2(rng.uniform(-75.0, 62.0, shape)).astype(np.float32)


@pytest.mark.parametrize("kind", ["unit", "steps", "wide"])
@pytest.mark.parametrize("shape,lb", [((2, 2, 2), 2), ((13, 13, 13), 2), ((33, 20, 33), 3), ((40, 40, 40), 3),
                                      ((33, 64, 31), 3), ((50, 35, 50), 4), ((240, 232, 240), 3)])
def test_gradients_match_the_formula(hip, kind, shape, lb):
    f = _field(kind, shape)
    with np.errstate(over="ignore"):
        g = np.gradient(f)
        norm = np.sqrt((g[0] * g[0] + g[1] * g[1]) + g[2] * g[2]) + np.float32(1e-8)
        ref = np.stack([x / norm for x in g], axis=-1)
    assert ref.dtype == np.float32
    c = _Context(hip, lb)
    try:
        v = c.volume(shape, "f32", "f32x3")
        v.upload_scalar_normals(f)
        s, n = v.download(scalar=True, normals=True)
        assert np.array_equal(s, f)
        assert np.array_equal(n == 0, ref == 0) and np.array_equal(np.signbit(n), np.signbit(ref))
        assert np.all(np.abs(n - ref) <= 3.6e-7 * np.abs(ref) + 2.0 ** -149)
    finally:
        c.close()
