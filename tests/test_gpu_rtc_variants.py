"""Tuning key 12: its default holds the bits that have an effect, and the others, which are accepted, change nothing:
the same passes run (bit for bit the same result, N = 528)."""
import numpy as np
import pytest

from lprec_amd import lpTransform
from lprec_amd._lib import LprecError

pytestmark = pytest.mark.gpu


def test_bits_without_effect(torch_cuda):
    torch = torch_cuda
    N0, P0, ns = 528, 60, 2
    print("case", N0, flush=True)
    lp = lpTransform(N0, P0, ns, "parzen", N0 / 2, "cubic")
    lp.precompute(0)
    lp.initcmem(0, 0)
    h = lp.clphandle[0]
    assert h.get_tuning(12) == 6
    R = torch.from_numpy(np.random.default_rng(12).standard_normal((ns, P0, N0)).astype(np.float32)).cuda()
    out = []
    for var in (6, 7, 14, 15):
        h.set_tuning(12, var)
        assert h.get_tuning(12) == var and h.get_tuning(10) == 1
        f = torch.full((ns, N0, N0), float("nan"), device="cuda")
        lp.adjp(f, R, 0)
        torch.cuda.synchronize()
        out.append(f)
    with pytest.raises(LprecError):
        h.set_tuning(12, 16)
    lp.close()
    for f in out[1:]:
        assert torch.equal(f, out[0])
