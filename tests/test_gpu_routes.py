"""Which way a call's cells are restricted: by strips of voxel faces or by
triangle lists, and with which caps."""
import ctypes

import numpy as np
import pytest

from meshes import icosphere

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,apex,strips", [(0, 1, True), (1, 1, True), (2, 1, False), (0, 0, False), (1, 0, False)])
def test_strip_room_is_for_strips(rpd, ctx, prec, apex, strips):
    """The larger cap that strips get (cells many voxels wide) is not for the
    triangle lists: the FP32 form, and the reference's corner apex."""
    x = rpd.generate_seeds(rpd.SEEDS_UNIFORM, 500, seed=3, wmax=0.0)
    dom = ctx.domain(rpd.Grid.voxels(np.ones(48 ** 3, np.uint8)))
    ctx.set_seeds(x)
    st = ctx.solve(dom, T=100, precision=prec, apex_mode=apex)
    dom.close()
    assert st["pass_caps"][0][3] == (min(1024, int(12 * (48 ** 3 / 500) ** (2 / 3))) if strips else 256)


@pytest.mark.parametrize("prec", [0, 1, 2])
@pytest.mark.parametrize("apex", [0, 1])
@pytest.mark.parametrize("kinds", ["all", "mesh and none", "voxel and none"])
def test_batch_of_both_kinds_of_domains(rpd, ctx, prec, apex, kinds):
    """A voxel domain, a mesh and no domain in one batch, each request as
    alone: the same bits, and over all passes (which pass counts a cell depends
    on the cap, the batch's largest) the same largest union of triangles."""
    P, T = icosphere(3, radius=2.0, rot_seed=11)
    doms = [ctx.domain(rpd.Grid.shape(rpd.SHAPE_SPHERE, 24, (0.5, 0.5, 0.5, 0.4))),
            ctx.domain(rpd.Grid.mesh(P, T, 40)), None]
    kinds = {"all": (0, 1, 2), "mesh and none": (1, 2), "voxel and none": (0, 2)}[kinds]
    reqs = [(doms[kinds[k % len(kinds)]], rpd.generate_seeds(rpd.SEEDS_UNIFORM, n, seed=n, wmax=0.0))
            for k, n in enumerate((5000, 3000, 700, 40, 20000, 17, 200))]
    caps = dict(precision=prec, apex_mode=apex, debug_counters=1)
    alone, status, most = [], [], 0

    def union():
        return max(ctx.debug_counters(p)["max"][3] for p in range(6))

    for d, x in reqs:
        ctx.set_seeds(x)
        ctx.solve(d, **caps)
        alone.append(ctx.moments())
        status.append(ctx.status())
        most = max(most, union())
    _, outs = ctx.solve_batch(reqs, **caps)
    got = ctx.status()
    assert union() == most
    for d in doms[:2]:
        d.close()
    assert np.array_equal(got, np.concatenate(status))
    for k, (o, m) in enumerate(zip(outs, alone)):
        assert np.array_equal(o, m, equal_nan=True), "request %d" % k


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("what", ["class", "open"])
def test_faces_that_do_not_bound_the_classes(rpd, ctx, prec, what):
    """Strips take another apex than the triangle lists, which is the same cell
    only if the faces are those between inside and outside voxels.  Where they
    are not (a class that says otherwise, a surface with holes) the result is
    that of the lists: of the same domain with a point off the lattice."""
    g, n = 8, 300
    x = rpd.generate_seeds(rpd.SEEDS_UNIFORM, n, seed=n, wmax=0.0)
    rng = np.random.default_rng(1)
    mask = np.ones((g, g, g), np.uint8)
    mask[2:6, 3:5, 1:4] = 0
    flips = rng.choice(g ** 3, 60, replace=False)
    ctx.set_seeds(x)
    out = []
    for off in (False, True):
        grid = rpd.Grid.voxels(mask.reshape(-1))
        d = grid.desc
        if what == "class":
            c = np.ctypeslib.as_array(ctypes.cast(d.centre, ctypes.POINTER(ctypes.c_int8)), (g ** 3,))
            c[flips] = 2 - c[flips]
        else:  # faces turned over: as many triangles, all in the lists
            t = np.ctypeslib.as_array(ctypes.cast(d.triangles, ctypes.POINTER(ctypes.c_int32)), (d.num_triangles, 3))
            k = rng.choice(d.num_triangles // 2, 40, replace=False) if not off else k
            for i in (2 * k, 2 * k + 1):
                t[i] = t[i][:, [1, 0, 2]]
        if off:
            p = ctypes.cast(d.points, ctypes.POINTER(ctypes.c_double))
            p[0] = np.nextafter(p[0], 500.0)
        dom = ctx.domain(grid)
        ctx.solve(dom, K=64, P=60, V=64, T=2000, precision=prec)
        out.append((ctx.moments(), ctx.status()))
        dom.close()
    v = 1e9 / n
    assert np.array_equal(out[0][1], out[1][1])
    assert np.abs(out[0][0][:, 3] - out[1][0][:, 3]).max() <= 1e-11 * v
