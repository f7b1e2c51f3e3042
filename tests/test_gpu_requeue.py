"""Re-queue passes of a solve: which form a cell's last pass has, and that no
pass repeats what cannot change."""
import numpy as np
import pytest

from meshes import icosphere

pytestmark = pytest.mark.gpu


def _sphere(m):
    """m directions, evenly spread."""
    k = np.arange(m) + 0.5
    z, a = 1 - 2 * k / m, np.pi * (1 + 5 ** 0.5) * k
    r = np.sqrt(1 - z * z)
    return np.stack((r * np.cos(a), r * np.sin(a), z), 1)


def _radius(u, d):
    """Largest vertex distance of the polytope {y: u_i . y <= d_i / 2}."""
    n = len(d)
    i, j, k = (t.reshape(-1) for t in np.meshgrid(*(np.arange(n),) * 3, indexing="ij"))
    keep = (i < j) & (j < k)
    i, j, k = i[keep], j[keep], k[keep]
    a = np.stack((u[i], u[j], u[k]), 1)
    ok = np.abs(np.linalg.det(a)) > 1e-9
    a, b = a[ok], np.stack((d[i], d[j], d[k]), 1)[ok] / 2
    y = np.linalg.solve(a, b[..., None])[..., 0]
    y = y[(y @ u.T <= d / 2 * (1 + 1e-12)).all(1)]
    return float(np.sqrt((y * y).sum(1).max()))


@pytest.mark.parametrize("steps", [2, 3])
@pytest.mark.parametrize("prec", [0, 1])
def test_the_last_step_has_no_margin(rpd, ctx, prec, steps):
    """One cell: its 60 faces overflow the planes in pass 1, the recomputation
    runs out of the 64 neighbours listed, and the 128th, the last that the next
    pass lists, lies between the cell's exact stop radius and the FP32 radius's
    margin over it.  The neighbours past the 60th lie behind others and cut
    nothing; those far out (their cells miss the domain) are there so that the
    list does not hold every seed."""
    m, D = 60, 200.0
    u = _sphere(m)
    d = D * (1 + 1e-3 * np.arange(m) / m)
    R = _radius(u, d)
    assert 2 * R > D * 1.03
    more = np.linspace(D * 1.005, D * 1.02, 67)
    v = u[np.arange(67) % m]
    last = 2 * R * (1 + 1e-5)
    far = _sphere(300)
    p = np.concatenate((np.zeros((1, 3)), u * d[:, None], v * more[:, None], u[:1] * last,
                        far * np.linspace(2.2 * D, 2.4 * D, 300)[:, None]))
    x = np.zeros((p.shape[0], 4))
    x[:, :3] = 500.0 + p
    mask = np.zeros((64, 64, 64), np.uint8)
    mask[31:33, 31:33, 31:33] = 1
    dom = ctx.domain(rpd.Grid.voxels(mask.reshape(-1)))
    ctx.set_seeds(x)
    st = ctx.solve(dom, K=64, P=50, V=256, precision=prec, max_extra_steps=steps)
    status, mom = ctx.status(), ctx.moments()
    dom.close()
    assert st["pass_cells"][:3] == [1, 1, 1]  # (the other cells miss the domain)
    assert [c[0] for c in st["pass_caps"][:3]] == [64, 64, 64]  # the third lists the 64 neighbours after those
    assert status[0] == 4
    assert abs(mom[0, 3] - 31.25 ** 3) < 1e-9 * 31.25 ** 3


@pytest.mark.parametrize("n", [10000, 100000])
def test_exact_failures_end_in_fp64(rpd, ctx, n):
    """The corner apex puts cone planes through lattice points, which leaves
    the cavities of some cells inconsistent in FP64.  The mixed form ends them
    with the FP64 form's status, and takes at most one pass more to find out."""
    x = rpd.generate_seeds(rpd.SEEDS_UNIFORM, n, seed=5, wmax=0.0)
    dom = ctx.domain(rpd.Grid.shape(rpd.SHAPE_TORUS, 100, (0.5, 0.5, 0.5, 0.3, 0.12)))
    ctx.set_seeds(x)
    out = []
    for prec in (0, 1):
        st = ctx.solve(dom, K=50, P=30, V=40, precision=prec, apex_mode=0)
        out.append((ctx.status(), st["passes"]))
    dom.close()
    assert (out[0][0] == 2).any()
    assert np.array_equal(out[0][0], out[1][0])
    assert out[1][1] <= out[0][1] + 1


@pytest.mark.parametrize("steps", [1, 5])
def test_overflows_do_not_see_other_requests_failures(rpd, ctx, steps):
    """Cells that meet more triangles than the cap finish in a second pass, in
    the form of the first; a batch's other request, whose cells fail the exact
    predicates there, changes none of their bits."""
    P, T = icosphere(4, radius=2.0, rot_seed=11)
    mesh = ctx.domain(rpd.Grid.mesh(P, T, 64))
    vox = ctx.domain(rpd.Grid.shape(rpd.SHAPE_SPHERE, 32, (0.5, 0.5, 0.5, 0.45)))
    x = rpd.generate_seeds(rpd.SEEDS_UNIFORM, 300, seed=1, wmax=0.0)
    y = rpd.generate_seeds(rpd.SEEDS_UNIFORM, 20000, seed=2, wmax=0.0)
    caps = dict(K=128, P=100, V=64, precision=1, apex_mode=0, max_extra_steps=steps)
    ctx.set_seeds(y)
    assert ctx.solve(vox, **caps)["fallback_cells"] > 0
    ctx.set_seeds(x)
    st = ctx.solve(mesh, **caps)
    alone, status = ctx.moments(), ctx.status()
    _, (got, _) = ctx.solve_batch([(mesh, x), (vox, y)], **caps)
    both = ctx.status()[:300]
    mesh.close()
    vox.close()
    assert st["passes"] > 1 and st["fallback_cells"] == 0 and st["pass_caps"][1][3] > st["pass_caps"][0][3]
    assert np.array_equal(status, both) and np.array_equal(got, alone)
