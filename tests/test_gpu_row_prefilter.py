"""The row prefilter (8 elements per lane, waves of 512, segments with halos)
where its cuts fall: rows of one wave (also the shortest and a full one), of
two and three segments, and images whose rows start at any float; and its
transpose by the dot test.  FP32 recursions with |z| < 0.27 keep a few
rounding errors of 6e-8 per sample: bound 1e-6 against FP64, and 1e-6 of
||A x|| ||y|| for the dot test (sums in FP64)."""
import numpy as np
import pytest

from lprec_amd import lpTransform
from oracle import mirror

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


@pytest.mark.parametrize("N0,interp", [(24, "cubic"), (101, "cubic"), (479, "cubic"), (512, "cubic"), (517, "cubic"),
                                       (965, "cubic"), (90, "linear"), (519, "linear")])
def test_rows(torch_cuda, N0, interp):
    torch = torch_cuda
    print("case", N0, interp, flush=True)
    P0, ns = 30, 2
    lp = lpTransform(N0, P0, ns, "none", N0 / 2 + 1.3, interp)
    lp.precompute(1)
    lp.initcmem(1, 0)
    h = lp.clphandle[0]
    tab = mirror.Tables(lp.glpars, lp.fwdparsi, lp.fwdparamsf, lp.adjparsi, lp.adjparamsf)
    N, P = tab.N, tab.Nproj
    rng = np.random.default_rng(N0)
    f = rng.standard_normal((ns, N0, N0)).astype(np.float32)
    R = rng.standard_normal((ns, P0, N0)).astype(np.float32)
    gf, gR = torch.from_numpy(f).cuda(), torch.from_numpy(R).cuda()
    of, oR = torch.zeros_like(gf), torch.zeros_like(gR)
    line = (lambda d: mirror.prefilter_line(d, -1)) if tab.cubic else (lambda d: d)
    o = N // 2 - N0 // 2
    d = np.zeros((ns, N, N))
    d[:, o:o + N0, o:o + N0] = f
    try:
        h.debug_stop(1)
        lp.fwdp(oR, gf, 0)
        a = h.debug_copy(4 if tab.cubic else 0, (ns, N, N))
        lp.adjp(of, gR, 0)
        b = h.debug_copy(4 if tab.cubic else 1, (ns, P, N))
    finally:
        h.debug_stop(0)
    keep = np.arange(P) % tab.os == 0 if tab.cubic else slice(None)
    e1, e2 = rel(a, line(d)), rel(b[:, keep], line(mirror.sino_prepare(tab, R))[:, keep])
    print("N %d rel image rows %.2e sinogram rows %.2e" % (N, e1, e2), flush=True)
    assert e1 <= 1e-6 and e2 <= 1e-6
    lp.fwdp(oR, gf, 0)
    lp.fwdp_transpose(of, gR, 0)
    torch.cuda.synchronize()
    lp.close()
    u, v = oR.cpu().numpy().astype(np.float64), of.cpu().numpy().astype(np.float64)
    assert abs((u * R).sum() - (f * v).sum()) <= 1e-6 * np.linalg.norm(u) * np.linalg.norm(R)
