"""Error against the FP64 oracle mirror at lengths whose compiled passes run radices 5, 10 and 20 (N = 1600: rows
5 16 10, columns 20 20 8; N = 2000: rows 10 10 10, columns 20 20 10).  Their constants, rounded one by one, have a
mean gain of up to 1e-7, more than all random rounding.  Bounds:
halfway between the error of the same inputs through the earlier stages of radices 2, 4, 5 and 8 (1600: fwd 1.25e-7,
adj 7.6e-8; 2000: 1.36e-7, 6.9e-8) and with those constants (1.38e-7, 1.00e-7; 1.51e-7, 1.12e-7)"""
import numpy as np
import pytest

from lprec_amd import lpTransform
from lprec_amd.phantom import phantom_stack

pytestmark = pytest.mark.gpu


def errors(torch, N0, P0=300, ns=2):
    from oracle import mirror
    print("case", N0, flush=True)
    lp = lpTransform(N0, P0, ns, "none", N0 / 2, "cubic")
    lp.precompute(1)
    lp.initcmem(1, 0)
    assert lp.clphandle[0].get_tuning(10) == 1
    f = phantom_stack(ns, N0, 12, seed=N0)
    R = torch.zeros((ns, P0, N0), device="cuda")
    g = torch.zeros((ns, N0, N0), device="cuda")
    lp.fwdp(R, torch.from_numpy(f).cuda(), 0)
    torch.cuda.synchronize()
    tab = mirror.Tables(lp.glpars, lp.fwdparsi, lp.fwdparamsf, lp.adjparsi, lp.adjparamsf)
    want = mirror.fwd(tab, f)
    data = want.astype(np.float32)
    lp.adjp(g, torch.from_numpy(data).cuda(), 0)
    torch.cuda.synchronize()
    back = mirror.adj(tab, data)
    lp.close()
    rel = lambda a, b: float(np.linalg.norm(a.cpu().numpy().astype(np.float64) - b) / np.linalg.norm(b))
    return rel(R, want), rel(g, back)


@pytest.mark.parametrize("N0,fwd,adj", [(1600, 1.32e-7, 8.8e-8), (2000, 1.43e-7, 9.1e-8)])
def test_no_gain_from_rounded_constants(torch_cuda, N0, fwd, adj):
    ef, ea = errors(torch_cuda, N0)
    print("N0 %d vs oracle: fwd %.3e adj %.3e" % (N0, ef, ea), flush=True)
    assert ef <= fwd and ea <= adj
