"""Which way a call's cells are restricted: by strips of voxel faces or by
triangle lists, and with which caps."""
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
def test_batch_of_both_kinds_of_domains(rpd, ctx, prec, apex):
    """A voxel domain, a mesh and no domain in one batch, each request as
    alone: the same bits, and over all passes (which pass counts a cell depends
    on the cap, the batch's largest) the same largest union of triangles."""
    P, T = icosphere(3, radius=2.0, rot_seed=11)
    doms = [ctx.domain(rpd.Grid.shape(rpd.SHAPE_SPHERE, 24, (0.5, 0.5, 0.5, 0.4))),
            ctx.domain(rpd.Grid.mesh(P, T, 40)), None]
    reqs = [(doms[k % 3], rpd.generate_seeds(rpd.SEEDS_UNIFORM, n, seed=n, wmax=0.0))
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
