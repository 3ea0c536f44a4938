"""Compiled passes whose LDS is close to the limit: N = 4608 (rows of 2304
points) against the generic kernels, adj with a filter.  Bound 2e-6, that of the
other lengths against the generic kernels, whose odd radices form the powers of
a root by recurrences."""
import numpy as np
import pytest

from lprec_amd import lpTransform

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [1, 3])
def test_rows_close_to_the_lds_limit(torch_cuda, ns):
    torch = torch_cuda
    N0, P0 = 4608, 48
    print("case", N0, ns, flush=True)
    lp = lpTransform(N0, P0, ns, "parzen", N0 / 2, "cubic")
    lp.precompute(0)
    lp.initcmem(0, 0)
    h = lp.clphandle[0]
    assert h.get_tuning(10) == 1
    R = torch.from_numpy(np.random.default_rng(ns).standard_normal((ns, P0, N0)).astype(np.float32)).cuda()
    out = []
    for compiled in (1, 0):
        h.set_tuning(10, compiled)
        f = torch.full((ns, N0, N0), float("nan"), device="cuda")
        lp.adjp(f, R, 0)
        torch.cuda.synchronize()
        out.append(f.double())
    lp.close()
    e = float((out[0] - out[1]).norm() / out[1].norm())
    print("compiled vs generic: %.2e" % e, flush=True)
    assert e <= 2e-6
