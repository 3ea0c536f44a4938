"""The transposes at every number of slices per launch where a kernel variant
starts (1, 2 and 5 for the box sums and the polar rows; 4 per block in the
polar columns; one more than a full group of 8), against the oracle's FP64
transposes slice by slice.  Bound 1e-5, that of the transposes' other oracle
tests (tables and sums in FP32).  The second geometry has few angles per
column and the third many, so that the polar columns' held and formed weights
both run."""
import numpy as np
import pytest

from lprec_amd import lpTransform
from oracle import mirror
from oracle import transpose as tr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N0,P0,interp", [(96, 80, "cubic"), (64, 48, "linear"), (64, 400, "cubic")])
def test_transposes_by_slices(torch_cuda, N0, P0, interp):
    torch = torch_cuda
    print("case", N0, P0, interp, flush=True)
    ns = 9
    lp = lpTransform(N0, P0, ns, "none", N0 / 2, interp)
    lp.precompute(1)
    lp.initcmem(1, 0)
    tab = mirror.Tables(lp.glpars, lp.fwdparsi, lp.fwdparamsf, lp.adjparsi, lp.adjparamsf)
    rng = np.random.default_rng(N0 + P0)
    R = rng.standard_normal((ns, P0, N0)).astype(np.float32)
    f = rng.standard_normal((ns, N0, N0)).astype(np.float32)
    cf, cR = tr.fwd_T(tab, R), tr.adj_T(tab, f, P0)
    gR, gf = torch.from_numpy(R).cuda(), torch.from_numpy(f).cuda()
    for n in (1, 2, 4, 5, 8, 9):
        a = torch.full((n, N0, N0), float("nan"), device="cuda")
        b = torch.full((n, P0, N0), float("nan"), device="cuda")
        lp.fwdp_transpose(a, gR[:n].contiguous(), 0)
        lp.adjp_transpose(b, gf[:n].contiguous(), 0)
        torch.cuda.synchronize()
        a, b = a.cpu().numpy(), b.cpu().numpy()
        for s in range(n):
            e1 = np.linalg.norm(a[s] - cf[s]) / np.linalg.norm(cf[s])
            e2 = np.linalg.norm(b[s] - cR[s]) / np.linalg.norm(cR[s])
            assert e1 <= 1e-5 and e2 <= 1e-5, (n, s, e1, e2)
    lp.close()
