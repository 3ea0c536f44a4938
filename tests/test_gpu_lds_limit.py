"""Mixed-radix kernels (tuning key 10 = 0) where their blocks come close to the 160 KB of LDS.  8 rows of 2400 points
and the static LDS beside them are 168712 bytes, so at N = 4800 a block takes 4; the filtered line pair of N = 5120
needs 168968 bytes of its own, so its call is refused, without a launch, and the handle stays usable.  Bound 2e-6
against the compiled passes, as at the other lengths with odd radices."""
import numpy as np
import pytest

from lprec_amd import lpTransform
from lprec_amd._lib import LprecError

pytestmark = pytest.mark.gpu


def _operator(N0, filt):
    print("case", N0, filt, flush=True)
    lp = lpTransform(N0, 48, 1, filt, N0 / 2, "cubic")
    lp.precompute(0)
    lp.initcmem(0, 0)
    return lp, lp.clphandle[0]


def _adj(torch, lp, R):
    f = torch.full((1, lp.N, lp.N), float("nan"), device="cuda")
    lp.adjp(f, R, 0)
    torch.cuda.synchronize()
    return f.double()


def _data(torch, N0):
    return torch.from_numpy(np.random.default_rng(N0).standard_normal((1, 48, N0)).astype(np.float32)).cuda()


def test_rows_leave_room_for_static_lds(torch_cuda):
    torch = torch_cuda
    lp, h = _operator(4800, "none")
    R = _data(torch, 4800)
    assert h.get_tuning(10) == 1
    a = _adj(torch, lp, R)
    h.set_tuning(10, 0)
    b = _adj(torch, lp, R)
    lp.close()
    e = float((a - b).norm() / b.norm())
    print("compiled vs generic: %.2e" % e, flush=True)
    assert e <= 2e-6


def test_a_block_over_the_limit_is_refused(torch_cuda):
    torch = torch_cuda
    lp, h = _operator(5120, "ramp")
    R = _data(torch, 5120)
    a = _adj(torch, lp, R)
    h.set_tuning(10, 0)
    with pytest.raises(LprecError):
        _adj(torch, lp, R)
    h.set_tuning(10, 1)
    assert torch.equal(_adj(torch, lp, R), a)
    lp.close()
