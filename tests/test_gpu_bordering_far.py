"""Bordering rings after a solve whose cells needed more neighbours than one
list holds (256): the unrestricted cells of the rings go on past a full list,
as a solve's do, and mark what the oracle marks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1, 2])
@pytest.mark.parametrize("n,K", [(300, 25), (600, 64), (1200, 25)])
def test_rings_past_a_full_list(rpd, orc, ctx, prec, n, K):
    # a ball of seeds, whose outer cells reach the frame's far side, and a lone
    # seed: their stop radius is never reached, so they use every seed
    rng = np.random.default_rng(n)
    x = np.zeros((n, 4))
    u = rng.normal(size=(n, 3))
    x[:, :3] = (250.0, 500.0, 500.0) + 60.0 * rng.random((n, 1)) ** (1 / 3) * u / np.linalg.norm(u, axis=1)[:, None]
    x[0, :3] = 850.0, 510.0, 490.0
    dom = ctx.domain(rpd.Grid.shape(rpd.SHAPE_CUBE, 16, ()))
    ctx.set_seeds(x)
    st = ctx.solve(dom, K=K, P=120, V=128, precision=prec, max_extra_steps=8)
    assert st["final_K"] > 256 and st["status_hist"][4] == n
    m = ctx.moments()
    dom.close()
    keep = 1e9 / n
    assert 0 < (m[:, 3] >= keep).sum() < n // 2
    for d in (0, 1, 2):
        out, ids = ctx.compact_used(keep, d)
        ref_out, ref_ids = orc.compact_used(x, m, keep, d, K=256, P=200, V=256, max_nb=200)
        assert np.array_equal(ids, ref_ids), d
        assert np.array_equal(out, ref_out), d
