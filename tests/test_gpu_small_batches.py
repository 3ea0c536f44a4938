"""Tile sizes, slices per block and the compiled passes' plans follow the batch
a handle is built for; the results of a slice may not: the operators and
their transposes from a one-slice handle against the slices of a batch, at
the grids where the rules switch (8-, 16-, 32- and 64-row tiles; 1, 2 and 4
slices per block), to FP32 rounding (bound 1e-6: the plans differ in the
order of the FFT's stages, the transposes sum per tile).  adj_T ends with the
FBP filter, which removes the mean that carries most of an image's energy
(ramp, 256 x 384: norm 163 before it, 0.74 after): the rounding of what
enters the filter is the scale there, i.e. the norm of the unfiltered adj_T
(the response is at most 1)."""
import pytest

from lprec_amd import lpTransform

pytestmark = pytest.mark.gpu


def rel(a, b, scale=None):
    return float((a.double() - b.double()).norm() / (b if scale is None else scale).double().norm())


@pytest.mark.parametrize("N0,P0,ns,filt,interp", [
    (64, 48, 9, "none", "cubic"),
    (101, 70, 5, "parzen", "cubic"),
    (256, 200, 4, "none", "linear"),
    (256, 384, 16, "ramp", "cubic"),
    (512, 384, 7, "none", "cubic"),
])
def test_slices_do_not_depend_on_the_batch(torch_cuda, N0, P0, ns, filt, interp):
    torch = torch_cuda
    print("case", N0, P0, ns, filt, interp, flush=True)
    g = torch.Generator(device="cuda").manual_seed(N0)
    f = torch.rand((ns, N0, N0), device="cuda", generator=g)
    R = torch.rand((ns, P0, N0), device="cuda", generator=g)
    out = []
    for batch in (ns, 1):
        lp = lpTransform(N0, P0, batch, filt, N0 / 2, interp)
        lp.precompute(1)
        lp.initcmem(1, 0)
        a, b, c, d = torch.zeros_like(R), torch.zeros_like(f), torch.zeros_like(f), torch.zeros_like(R)
        for s in range(0, ns, batch):
            e = s + batch
            lp.fwdp(a[s:e], f[s:e], 0)
            lp.adjp(b[s:e], R[s:e], 0)
            lp.fwdp_transpose(c[s:e], R[s:e], 0)
            lp.adjp_transpose(d[s:e], f[s:e], 0)
        torch.cuda.synchronize()
        lp.close()
        out.append((a, b, c, d))
    (a, b, c, d), (a1, b1, c1, d1) = out
    print("fwd %.1e adj %.1e fwd_T %.1e adj_T %.1e" % (rel(a1, a), rel(b1, b), rel(c1, c), rel(d1, d)), flush=True)
    assert torch.isfinite(a).all() and torch.isfinite(b).all()
    assert rel(a1, a) <= 1e-6 and rel(b1, b) <= 1e-6 and rel(c1, c) <= 1e-6
    scale = None
    if filt != "none":
        lp = lpTransform(N0, P0, ns, "none", N0 / 2, interp)
        lp.precompute(0)
        lp.initcmem(0, 0)
        scale = torch.zeros_like(R)
        lp.adjp_transpose(scale, f, 0)
        torch.cuda.synchronize()
        lp.close()
    assert rel(d1, d, scale) <= 1e-6
