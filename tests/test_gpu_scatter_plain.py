"""The tiled scatter on tiles without a colouring, which k_scatter adds with LDS atomics while k_scatter_col has the
others: the transpose of the polar gather forced onto the tiles (key 7 = 0) against the oracle on the same tables.  The
precomputed tables need at most 256 colour classes per tile; here their rho coordinates are drawn together by 4, which
takes up to 4 times as many (on tiles of 32 and 64 rows, i.e. from 7 slices on).  A point of the grid collects up to
~4000 FP32 terms in an unordered sum: 6e-8 sqrt(4000) = 4e-6 of its magnitude at most, bound 1e-5 as for the other
transposes."""
import re

import numpy as np
import pytest

from lprec_amd import lpTransform
from oracle import mirror
from oracle import transpose as tr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns,interp", [(7, "cubic"), (15, "cubic"), (7, "linear")])
def test_uncoloured_tiles(torch_cuda, monkeypatch, capfd, ns, interp):
    torch = torch_cuda
    N0, P0 = 64, 600
    monkeypatch.setenv("LPREC_AMD_VERBOSE", "1")
    lp = lpTransform(N0, P0, ns, "none", N0 / 2, interp)
    lp.precompute(1)
    points = int(sum(lp.fwdparsi[:3]))
    first = 6 * int(lp.fwdparsi[3 + points]) + points   # after the image coordinates and the theta ones
    rho = lp.fwdparamsf[first:first + points]
    rho[:] = np.float32(rho.mean()) + (rho - np.float32(rho.mean())) / 4
    lp.initcmem(1, 0)
    tiles, coloured = map(int, re.search(r"log-polar->polar: (\d+) tiles, (\d+) coloured", capfd.readouterr().err).groups())
    print("case", ns, interp, "tiles", tiles, "coloured", coloured, flush=True)
    assert coloured < tiles
    R = np.random.default_rng(ns).standard_normal((ns, P0, N0)).astype(np.float32)
    want = tr.fwd_T(mirror.Tables(lp.glpars, lp.fwdparsi, lp.fwdparamsf, lp.adjparsi, lp.adjparamsf), R)
    h, gR = lp.clphandle[0], torch.from_numpy(R).cuda()
    h.set_tuning(7, 0)
    f = torch.full((ns, N0, N0), float("nan"), device="cuda")
    lp.fwdp_transpose(f, gR, 0)
    torch.cuda.synchronize()
    e = float(np.linalg.norm(f.cpu().numpy() - want) / np.linalg.norm(want))
    print("rel %.1e" % e, flush=True)
    assert e <= 1e-5
    lp.close()
