"""What a handle's plan of the compiled passes does: rows whose LDS is close to the limit, and what the tuning
keys of these passes read back and run.  N = 4608 (rows of 2304 points) against the generic kernels, adj with a
filter: bound 2e-6, that of the other lengths against the generic kernels, whose odd radices form the powers of a root
by recurrences."""
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


@pytest.mark.parametrize("N0,loaded", [
    (2064, 1),
    (6864, 0),   # no plan for the columns (13728 points: radix 13 alone has more butterflies than threads)
])
def test_key_10_tells_whether_every_pass_is_compiled(torch_cuda, N0, loaded):
    print("case", N0, flush=True)
    lp = lpTransform(N0, 48, 1, "none", N0 / 2, "cubic")
    lp.precompute(0)
    lp.initcmem(0, 0)
    got = lp.clphandle[0].get_tuning(10)
    lp.close()
    assert got == loaded


@pytest.mark.parametrize("N0,ns", [(80, 2), (528, 8)])
def test_threads_of_the_column_pass(torch_cuda, N0, ns):
    """Key 11: every accepted count runs, reads back, and gives the automatic one's result (1e-6: the radices may
    come in another order)."""
    torch = torch_cuda
    print("case", N0, ns, flush=True)
    lp = lpTransform(N0, 60, ns, "none", N0 / 2, "cubic")
    lp.precompute(0)
    lp.initcmem(0, 0)
    h = lp.clphandle[0]
    R = torch.from_numpy(np.random.default_rng(N0).standard_normal((ns, 60, N0)).astype(np.float32)).cuda()
    out = []
    for threads in (0, 256, 512, 1024):
        h.set_tuning(11, threads)
        assert h.get_tuning(10) == 1 and (h.get_tuning(11) == threads or not threads)
        f = torch.full((ns, N0, N0), float("nan"), device="cuda")
        lp.adjp(f, R, 0)
        torch.cuda.synchronize()
        out.append(f.double())
    lp.close()
    for f in out[1:]:
        assert float((f - out[0]).norm() / out[0].norm()) <= 1e-6
