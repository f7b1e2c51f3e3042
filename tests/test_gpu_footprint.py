"""What a server counts a request with, against the device memory that a
context holds once it has solved it."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,P,V,steps,prec", [(25, 35, 40, 5, 1), (20, 30, 40, 1, 1), (20, 30, 40, 1, 0),
                                              (30, 30, 40, 1, 2), (25, 35, 40, 5, 2), (64, 40, 60, 5, 1),
                                              (64, 40, 100, 5, 0), (10, 30, 40, 2, 1), (50, 32, 48, 0, 0)])
def test_a_request_holds_what_it_is_counted_with(rpd, ctx, K, P, V, steps, prec):
    n = 200000
    count = rpd.lib().rpd_solve_bytes
    count.restype, count.argtypes = ctypes.c_int64, [ctypes.c_int64, ctypes.c_void_p]
    p = rpd.params(K=K, P=P, V=V, precision=prec, max_extra_steps=steps)
    x = rpd.generate_seeds(rpd.SEEDS_UNIFORM, n, seed=5, wmax=0.0)
    dom = ctx.domain(rpd.Grid.shape(rpd.SHAPE_CUBE, 32, ()))
    ctx.set_seeds(x[:1000])
    ctx.solve(dom, K=K, P=P, V=V, precision=prec)  # the kernels' code is loaded
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    c = rpd.Context(0)
    c.solve_batch([(dom, x)], K=K, P=P, V=V, precision=prec, max_extra_steps=steps)
    torch.cuda.synchronize()
    held = free - torch.cuda.mem_get_info()[0]
    c.close()
    dom.close()
    counted = count(n, ctypes.byref(p))
    print("footprint", K, P, V, steps, prec, "held %.0f counted %.0f bytes a seed" % (held / n, counted / n), flush=True)
    assert 0 < held <= counted
