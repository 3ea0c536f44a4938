"""The row, column and filtered-sinogram passes compiled at run time, over the
kinds of length their plans distinguish: register radices only (smooth
lengths, from the smallest grid up), one matrix-core stage (a prime factor
17 .. 263: one to nine output tiles, with and without a remainder of the
16-wide tiles and 4-deep steps), two of them (17 x 17, the second with
twiddles), several slices per block, and no data outside a row band.

Bounds, from FP32 rounding (eps 6e-8, ~20 rounded operations deep per
transform, four transforms): 1e-6 against the FP64 oracle mirror.  Against the
generic kernels 2e-6: those form the powers of an odd radix's root by
recurrences of up to 7 products (4e-7 each) in all four transforms.
"""
import numpy as np
import pytest

from lprec_amd import lpTransform
from lprec_amd.phantom import phantom_stack

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


def _lp(N0, P0, ns, filt, cor, interp, fwd):
    lp = lpTransform(N0, P0, ns, filt, cor, interp)
    lp.precompute(fwd)
    lp.initcmem(fwd, 0)
    assert lp.clphandle[0].get_tuning(10) == 1, "no compiled passes at N0 = %d" % N0
    return lp


def _run(lp, f, R, torch):
    out = []
    if f is not None:
        Ro = torch.zeros((f.shape[0], lp.Nproj, lp.N), device="cuda")
        lp.fwdp(Ro, torch.from_numpy(f).cuda(), 0)
        out.append(Ro)
    fo = torch.zeros((R.shape[0], lp.N, lp.N), device="cuda")
    lp.adjp(fo, torch.from_numpy(R).cuda(), 0)
    out.append(fo)
    torch.cuda.synchronize()
    return [o.cpu().numpy() for o in out]


@pytest.mark.parametrize("N0,P0,ns,filt,cor,interp", [
    (64, 48, 2, "parzen", 32, "cubic"),      # h = 32, rho 128, filter 128: the smallest grid
    (80, 60, 1, "none", 40, "cubic"),        # factor 5
    (141, 70, 2, "ramp", 71.2, "linear"),    # N = 144 = 2^4 3^2, odd width
    (176, 90, 1, "hamming", 88, "cubic"),    # factor 11
    (208, 90, 1, "none", 104, "cubic"),      # factor 13
    (272, 120, 3, "parzen", 136, "cubic"),   # 17: 9 outputs, one tile, 9 terms
    (304, 120, 1, "none", 152, "cubic"),     # 19
    (496, 180, 1, "ramp", 248, "cubic"),     # 31: 16 outputs, exactly one tile
    (526, 180, 2, "none", 263.4, "cubic"),   # N = 528: register radices 22 and 24
    (417, 120, 11, "parzen", 208.5, "cubic"),# N = 432: 216 points as 18 x 12, slices in turn
    (592, 200, 1, "none", 296, "linear"),    # 37: 19 outputs, two tiles
    (752, 240, 1, "parzen", 376, "cubic"),   # 47: 24 terms, six full steps
])
def test_compiled_lengths_match_oracle(torch_cuda, N0, P0, ns, filt, cor, interp):
    from oracle import mirror
    print("case", N0, P0, ns, filt, cor, interp, flush=True)
    f = phantom_stack(ns, N0, 12, seed=N0)
    R = np.random.default_rng(N0).standard_normal((ns, P0, N0)).astype(np.float32)
    lp = _lp(N0, P0, ns, filt, cor, interp, 1)
    got = _run(lp, f, R, torch_cuda)
    tab = mirror.Tables(lp.glpars, lp.fwdparsi, lp.fwdparamsf, lp.adjparsi, lp.adjparamsf)
    ef, ea = rel(got[0], mirror.fwd(tab, f)), rel(got[1], mirror.adj(tab, R))
    print("N0 %d vs oracle: fwd %.2e adj %.2e" % (N0, ef, ea), flush=True)
    assert ef <= 1e-6 and ea <= 1e-6


@pytest.mark.parametrize("N0,P0,ns,filt", [
    (1072, 64, 2, "none"),     # 67: three output tiles
    (1168, 64, 1, "parzen"),   # 73
    (2064, 64, 12, "none"),    # 43, several slices per row block
    (2096, 64, 2, "parzen"),   # 131: five tiles
    (2128, 64, 1, "none"),     # 7 x 19
    (4208, 48, 1, "none"),     # 263: nine tiles
    (4624, 48, 1, "none"),     # 17 x 17: a matrix-core stage with twiddles
])
def test_compiled_lengths_match_generic(torch_cuda, N0, P0, ns, filt):
    print("case", N0, P0, ns, filt, flush=True)
    R = np.random.default_rng(N0).standard_normal((ns, P0, N0)).astype(np.float32)
    lp = _lp(N0, P0, ns, filt, N0 / 2, "cubic", 0)
    a = _run(lp, None, R, torch_cuda)[0]
    h = lp.clphandle[0]
    h.set_tuning(10, 0)
    b = _run(lp, None, R, torch_cuda)[0]
    h.set_tuning(10, 1)
    e = rel(a, b)
    print("N0 %d compiled vs generic: %.2e" % (N0, e), flush=True)
    assert e <= 2e-6
