"""What precedes a solve's kNN, at the edges of its tiles: the binning's scan
(2,048 cells a workgroup, sums of up to 64 earlier workgroups read at once) and
the list of the cells that the cover test keeps (1,024 seeds a workgroup).
Both are whole numbers: exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cells(x, dim, real):
    c = np.floor(x[:, :3].astype(real) * real(dim) / real(1000.0)).astype(np.int64).clip(0, dim - 1)
    return c[:, 0] + c[:, 1] * dim + c[:, 2] * dim * dim


@pytest.mark.parametrize("prec,real", [(0, np.float64), (1, np.float32)])
@pytest.mark.parametrize("n", [2, 5500, 7000, 406000, 450001])
def test_binning_is_the_stable_sort(rpd, ctx, prec, real, n):
    # dim^3 + 1 cells: 2, 1729 and 2198 (one tile, two), 64 and 70 tiles
    x = rpd.generate_seeds(rpd.SEEDS_UNIFORM, n, seed=n, wmax=0.0)
    dim = max(1, int(np.floor(np.cbrt(n / 3.1) + 0.5)))
    ctx.set_seeds(x)
    ctx.solve(None, K=min(4, n - 1), P=40, V=60, precision=prec, max_extra_steps=0)
    assert np.array_equal(ctx.perm(), np.argsort(_cells(x, dim, real), kind="stable"))


@pytest.mark.parametrize("n", [1023, 1024, 1025, 66000, 140001])
def test_kept_cells_are_the_whole_diagram(rpd, ctx, n):
    h = (1.0 / n) ** (1 / 3)
    x = rpd.generate_seeds(rpd.SEEDS_UNIFORM, n, seed=n, wmax=0.25 * h * h * 1e6)
    dom = ctx.domain(rpd.Grid.shape(0, 32, (0.5, 0.5, 0.5, 0.2)))
    ctx.set_seeds(x)
    out = []
    for cull in (1, 0):
        st = ctx.solve(dom, K=64, P=48, V=64, precision=1, cull=cull)
        out.append((ctx.moments(), st["skipped_cells"], st["pass_cells"][0]))
    dom.close()
    assert out[0][1] > 0 and out[0][1] + out[0][2] == n and out[1][1] == 0
    assert np.array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("crowded", [False, True])
def test_batch_is_binned_as_alone(rpd, ctx, prec, crowded):
    """The requests' binnings in one go: each request's permutation and weight
    minima as alone, also when a cell of one of them holds more seeds than a
    run that is sorted in place."""
    rng = np.random.default_rng(5)
    reqs = []
    for k, n in enumerate((2, 700, 3001, 40000, 17)):
        x = rpd.generate_seeds(rpd.SEEDS_UNIFORM, n, seed=n, wmax=10.0 * k)
        if crowded and n == 3001:
            x[:200, :3] = 300.0 + rng.random((200, 3))
        reqs.append(x)
    dom = ctx.domain(rpd.Grid.shape(0, 24, (0.5, 0.5, 0.5, 0.4)))
    caps = dict(K=64, P=48, V=64, precision=prec)
    alone, perms = [], []
    base = 0
    for x in reqs:
        ctx.set_seeds(x)
        ctx.solve(dom, **caps)
        alone.append(ctx.moments())
        perms.append(ctx.perm() + base)
        base += x.shape[0]
    _, outs = ctx.solve_batch([(dom, x) for x in reqs], **caps)
    perm = ctx.perm()
    dom.close()
    assert np.array_equal(perm, np.concatenate(perms))
    for k, (o, m) in enumerate(zip(outs, alone)):
        assert np.array_equal(o, m), "request %d" % k


@pytest.mark.parametrize("prec", [0, 1, 2])
@pytest.mark.parametrize("K,steps,reach", [(20, 1, 40), (7, 2, 28), (30, 2, 120)])
def test_neighbours_in_all_are_what_the_caps_allow(rpd, ctx, prec, K, steps, reach):
    """However the first list is sized, a cell may use K neighbours, doubled
    once a pass: the cells that run out are those of one list of that length
    (the FP32 form goes on in FP64)."""
    x = rpd.generate_seeds(rpd.SEEDS_UNIFORM, 3000, seed=9, wmax=0.0)
    x[:, :3] = 200.0 + 0.6 * x[:, :3]  # cells of the outer seeds reach far
    dom = ctx.domain(rpd.Grid.shape(0, 16, (0.5, 0.5, 0.5, 0.45)))
    ctx.set_seeds(x)
    ctx.solve(dom, K=K, P=100, V=128, precision=prec, max_extra_steps=steps)
    got = ctx.status()
    ctx.solve(dom, K=reach, P=100, V=128, precision=0, max_extra_steps=0)
    ref = ctx.status()
    dom.close()
    assert (ref != 4).any()
    assert np.array_equal(got, ref)
