"""Soundness of the mixed form's filter with the bound the kernels use (CPU
only): kappa * ((|e.x| + |e.y| + |e.z|) M + |e.w| 1.1548), M = |w1| + |w2| +
|w3| of the vertex's three planes.  Over near-degenerate configurations,
evaluated in FP32 as the kernels do, with and without fused multiply-adds,
every sign outside the bound is the exact one of the FP64 planes, so every
wrong sign is left to FP64."""
import numpy as np
import pytest

from test_filter_bound import KAPPA, _exact_sign, _fp32_eval, _plane

MAG_W = np.float32(1.1548)


def _bound(p1, p2, p3, e):
    f = np.float32
    m = abs(f(p1[3])) + abs(f(p2[3])) + abs(f(p3[3]))
    ek = f(KAPPA) * (abs(f(e[0])) + abs(f(e[1])) + abs(f(e[2])))
    ewk = f(KAPPA) * MAG_W * abs(f(e[3]))
    return float(f(np.float64(ek) * np.float64(m) + np.float64(ewk)))  # one fused multiply-add


@pytest.mark.parametrize("seed,squeeze", [(1, 1.0), (2, 1e-1), (3, 4e-2)])
def test_no_wrong_sign_is_trusted(seed, squeeze):
    """squeeze: how far apart the three normals are (|W| is about its square;
    below 1e-3 every test of a vertex is left to FP64)."""
    rng = np.random.default_rng(seed)
    trusted = open_ = wrong = 0
    for it in range(2500):
        scale = 10.0 ** rng.uniform(0, 2.5)
        p1 = _plane(rng, scale)
        others = []
        for _ in range(2):
            q = _plane(rng, scale)
            q[:3] = p1[:3] + squeeze * q[:3] if squeeze < 1 else q[:3]
            q[:3] /= np.linalg.norm(q[:3])
            others.append(q)
        p2, p3 = others
        a = np.array([p1[:3], p2[:3], p3[:3]])
        if abs(np.linalg.det(a)) < 1e-9:
            continue
        v = np.linalg.solve(a, -np.array([p1[3], p2[3], p3[3]]))
        n = rng.normal(size=3)
        n /= np.linalg.norm(n)
        off = 10.0 ** rng.uniform(-9, 0) * scale * rng.choice([-1.0, 1.0])
        e = np.array([n[0], n[1], n[2], -(n @ v) + off])
        exact = _exact_sign(p1, p2, p3, e)
        bound = _bound(p1, p2, p3, e)
        for fused in (False, True):
            sv = _fp32_eval(p1, p2, p3, e, fused)[0]
            right = (sv > 0) - (sv < 0) == exact
            if abs(sv) > bound:
                trusted += 1
                assert right, (it, fused, sv, bound)
            else:
                open_ += 1
                wrong += not right
    assert trusted > 100 and open_ > 100 and wrong > 10
