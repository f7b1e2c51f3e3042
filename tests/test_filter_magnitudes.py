"""The magnitudes the mixed form's filter bounds its error with (CPU only).

The filter's error bound is kappa times the sums of |terms| of the cofactors
X, Y, Z and W.  The kernel takes |w1| + |w2| + |w3| for the first three and
1.1548 (above 2 / sqrt(3)) for W.  For planes with unit normals, rounded to
FP32 as the kernel holds them, both must be at least the sums, up to the
rounding of the normals (2^-22 of the bound; the factor kappa is 64 units
where first-order analysis gives 13).
"""
import numpy as np
import pytest


def _sums(p1, p2, p3):
    a = np.abs
    ab = lambda i, j: a(p2[..., i] * p3[..., j]) + a(p2[..., j] * p3[..., i])  # noqa: E731
    x, y, z, w = (a(p1[..., i]) for i in range(4))
    mx = w * ab(1, 2) + y * ab(2, 3) + z * ab(1, 3)
    my = x * ab(2, 3) + w * ab(0, 2) + z * ab(0, 3)
    mz = x * ab(1, 3) + y * ab(0, 3) + w * ab(0, 1)
    return np.maximum(mx, np.maximum(my, mz)), x * ab(1, 2) + y * ab(0, 2) + z * ab(0, 1)


@pytest.mark.parametrize("spread", [1.0, 1e-2, 1e-5])
def test_magnitudes_bound_the_sums(spread):
    rng = np.random.default_rng(7)
    n = 200000
    base = rng.normal(size=(n, 1, 3))
    v = base + spread * rng.normal(size=(n, 3, 3))  # from unrelated normals to nearly parallel ones
    v[: n // 10] = np.sign(v[: n // 10])            # the normals that reach the bound of W
    v /= np.linalg.norm(v, axis=2, keepdims=True)
    w = rng.uniform(-1, 1, size=(n, 3, 1)) * 10.0 ** rng.uniform(-6, 3, size=(n, 3, 1))
    p = np.concatenate((v, w), 2).astype(np.float32).astype(np.float64)
    mxyz, mw = _sums(p[:, 0], p[:, 1], p[:, 2])
    slack = 1 + 2.0 ** -22
    assert (mxyz <= np.abs(p[:, :, 3]).sum(1) * slack).all()
    assert (mw <= 1.1548).all()
    assert mw.max() > 1.1547 - 1e-3
