"""The streaming column pass at every power-of-two length (rho 256 .. 4096):
shared waves (4 and 2 frequencies), one to several columns per block and spans
that end inside a block's run of columns.  The input is a constant plus noise, so the
packed theta-DC / Nyquist frequency carries most of the energy.  Bound 1e-6
against the FP64 oracle mirror (four FP32 transforms, eps 6e-8)."""
import numpy as np
import pytest

from lprec_amd import lpTransform

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


@pytest.mark.parametrize("N0,P0,ns,check", [
    (128, 96, 5, (0, 4)),       # rho 256: four frequencies per wave
    (256, 120, 3, (0, 2)),      # rho 512: two
    (512, 150, 11, (0, 7, 10)), # rho 1024, several columns per block
    (1024, 90, 5, (0, 4)),      # rho 2048
    (2048, 60, 7, (0, 6)),      # rho 4096: 21 columns in runs that cross the spans
])
def test_column_pass_matches_oracle(torch_cuda, N0, P0, ns, check):
    torch = torch_cuda
    from oracle import mirror
    print("case", N0, P0, ns, flush=True)
    rng = np.random.default_rng(N0)
    f = (1.0 + 0.1 * rng.standard_normal((ns, N0, N0))).astype(np.float32)
    R = (1.0 + 0.1 * rng.standard_normal((ns, P0, N0))).astype(np.float32)
    lp = lpTransform(N0, P0, ns, "none", N0 / 2, "cubic")
    lp.precompute(1)
    lp.initcmem(1, 0)
    Ro = torch.zeros((ns, P0, N0), device="cuda")
    fo = torch.zeros((ns, N0, N0), device="cuda")
    lp.fwdp(Ro, torch.from_numpy(f).cuda(), 0)
    lp.adjp(fo, torch.from_numpy(R).cuda(), 0)
    torch.cuda.synchronize()
    tab = mirror.Tables(lp.glpars, lp.fwdparsi, lp.fwdparamsf, lp.adjparsi, lp.adjparamsf)
    at = list(check)
    ef = rel(Ro.cpu().numpy()[at], mirror.fwd(tab, f[at]))
    ea = rel(fo.cpu().numpy()[at], mirror.adj(tab, R[at]))
    print("N0 %d: fwd %.2e adj %.2e" % (N0, ef, ea), flush=True)
    assert ef <= 1e-6 and ea <= 1e-6


@pytest.mark.parametrize("ns", [1, 2])
def test_column_pass_8192_matches_mixed_radix(torch_cuda, ns):
    """rho 8192 (32 x 16 x 16): against the mixed-radix kernels (family 0), 3
    and 6 columns per frequency; the same input and bound."""
    torch = torch_cuda
    print("case 4096", ns, flush=True)
    N0, P0 = 4096, 48
    g = torch.Generator(device="cuda").manual_seed(ns)
    f = 1.0 + 0.1 * torch.randn((ns, N0, N0), device="cuda", generator=g)
    R = 1.0 + 0.1 * torch.randn((ns, P0, N0), device="cuda", generator=g)
    lp = lpTransform(N0, P0, ns, "none", N0 / 2, "cubic")
    lp.precompute(1)
    lp.initcmem(1, 0)
    out = []
    for family in (2, 0):
        lp.clphandle[0].set_tuning(4, family)
        a, b = torch.full_like(R, float("nan")), torch.full_like(f, float("nan"))
        lp.fwdp(a, f, 0)
        lp.adjp(b, R, 0)
        torch.cuda.synchronize()
        out.append((a, b))
    lp.close()
    for x, y in zip(*out):
        e = float((x.double() - y.double()).norm() / y.double().norm())
        print("rel %.1e" % e, flush=True)
        assert e <= 1e-6
