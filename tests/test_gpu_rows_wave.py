"""The inverse row pass with 32 elements per lane at h = 1024 and 2048 against
the radix-16 register kernels (FFT kernel family 1), forward and adjoint, for
one slice and for slice counts that the slices per block do not divide.  Both
are FP32 transforms of 2048 or 4096 points: a relative difference of a few
1e-8 per pass, bound 1e-6."""
import pytest

from lprec_amd import lpTransform

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N0,ns", [(2048, 1), (2048, 5), (4096, 1), (4096, 3)])
def test_inverse_rows(torch_cuda, N0, ns):
    torch = torch_cuda
    print("case", N0, ns, flush=True)
    P0 = 48
    g = torch.Generator(device="cuda").manual_seed(N0 + ns)
    f = torch.rand((ns, N0, N0), device="cuda", generator=g)
    R = torch.rand((ns, P0, N0), device="cuda", generator=g)
    lp = lpTransform(N0, P0, ns, "none", N0 / 2, "cubic")
    lp.precompute(1)
    lp.initcmem(1, 0)
    out = []
    for family in (2, 1):
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
