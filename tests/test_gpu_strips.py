"""Restriction by voxel-face strips against the triangle lists.

A domain made of voxel faces whose voxel classes are all known is restricted
by strips of faces; with one point of it a unit in the last place off the
lattice, it takes the general triangle lists (with another cone apex per
cell).  Both cut the same cells by the same domain, so moments and faces
differ by rounding only: each of the two sums a few hundred pieces of at most
the cell's volume, whose FP64 rounding stays below 1e-13 of the mean cell
apiece, so 1e-11 of the mean cell volume bounds the difference (faces: 1e-10
of a face's scale, as areas are an order lower).
"""
import ctypes

import numpy as np
import pytest

from conftest import moment_errors

pytestmark = pytest.mark.gpu


def _mask(kind, g):
    rng = np.random.default_rng(g)
    if kind == "full":
        return np.ones(g ** 3, np.uint8)
    if kind == "random":  # isolated voxels, edges and corners shared by two
        return (rng.random(g ** 3) < 0.5).astype(np.uint8)
    m = np.zeros((g, g, g), np.uint8)  # slabs and bars: runs that end inside and at the frame
    m[: g // 2] = 1
    m[:, g // 3: g // 3 + 1, :] = 1
    m[g // 2:, :, g - 1] = 1
    return m.reshape(-1)


@pytest.mark.parametrize("kind,g,n", [("full", 1, 40), ("full", 5, 900), ("random", 2, 60), ("random", 7, 4000),
                                      ("random", 23, 50), ("slabs", 12, 700), ("slabs", 33, 30)])
@pytest.mark.parametrize("prec", [0, 1])
def test_strips_match_triangle_lists(rpd, ctx, kind, g, n, prec):
    h = (1.0 / n) ** (1 / 3)
    x = rpd.generate_seeds(rpd.SEEDS_UNIFORM, n, seed=n, wmax=0.25 * h * h * 1e6)
    # seeds on lattice planes and at the frame's corner
    x[: n // 4, 0] = np.round(x[: n // 4, 0] * g / 1000.0) * (1000.0 / g)
    x[0, :3] = 0.0
    grid = rpd.Grid.voxels(_mask(kind, g))
    lists = rpd.Grid.voxels(_mask(kind, g))
    point = ctypes.cast(lists.desc.points, ctypes.POINTER(ctypes.c_double))
    point[0] = np.nextafter(point[0], 500.0)
    ctx.set_seeds(x)
    out = []
    for d in (grid, lists):
        dom = ctx.domain(d)
        st = ctx.solve(dom, K=64, P=60, V=64, T=4000, precision=prec, H=64, HC=4)
        faces, ids = ctx.hessian()
        withh = ctx.moments()
        ctx.solve(dom, K=64, P=40, V=60, T=100, precision=prec)
        out.append((ctx.moments(), withh, ctx.status(), faces, ids, st))
        dom.close()
    (m0, h0, s0, f0, i0, st0), (m1, h1, s1, f1, i1, _) = out
    ev, em = moment_errors(m0, m1, n)
    eh = max(moment_errors(h0, h1, n))
    print("strips", kind, g, n, prec, st0["passes"], "%.2e %.2e %.2e" % (ev, em, eh), flush=True)
    vol = grid.volume()
    assert abs(m0[:, 3].sum() - vol) / vol < 1e-11
    assert np.array_equal(s0, s1)
    assert max(ev, em, eh) <= 1e-11
    face = 1e6 * h * h
    same = (i0 == i1).all(1)
    # a neighbour may differ only where a face's area is at the 0.2 threshold
    assert (~same).sum() <= n // 100
    assert np.abs(f0[same][:, :, 3] - f1[same][:, :, 3]).max() <= 1e-10 * face
    assert np.abs(f0[same][:, :, :3] - f1[same][:, :, :3]).max() <= 1e-10 * face * 1000.0


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("g,n", [(24, 6), (16, 40)])
def test_strip_cap_does_not_change_cells(rpd, ctx, g, n, prec):
    """Cells that meet more strips than the cap take a pass over the same
    records with a larger one; batches of strips are the same for every cap
    and number of waves: the same bits as with room from the beginning."""
    x = rpd.generate_seeds(rpd.SEEDS_UNIFORM, n, seed=n, wmax=0.0)
    dom = ctx.domain(rpd.Grid.voxels(_mask("random", g)))
    ctx.set_seeds(x)
    out = []
    for T in (10, 1500, 20000):
        st = ctx.solve(dom, K=64, P=60, V=64, T=T, precision=prec)
        out.append((ctx.moments(), ctx.status(), st["passes"]))
    dom.close()
    assert out[0][2] > out[2][2], "no cell above the smallest cap"
    for m, s, _ in out[1:]:
        assert np.array_equal(m, out[0][0]) and np.array_equal(s, out[0][1])
