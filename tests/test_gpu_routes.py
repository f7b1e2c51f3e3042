"""Which way a call's cells are restricted: by strips of voxel faces or by
triangle lists, and with which caps."""
import numpy as np
import pytest

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
