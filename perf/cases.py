"""The calls that users of this package make, as measured cases: single operator calls from the smallest grids to
the largest, one slice and whole batches, centred scans and scans whose centre pads the grid to an awkward length,
filtered and unfiltered, cubic and linear, with gradients, and one whole iterative reconstruction.

A case names the operator (``op``), the geometry and the batch:

* ``fwd``   R = lp.fwdp(f)                      * ``adj``   f = lp.adjp(R), with the FBP filter if there is one
* ``radon`` a data-fit step: R = radon(f) and the gradient of ||R - g||^2 with respect to f
* ``bproj`` the same through backprojection(R): the image and the gradient of ||f - g||^2 with respect to R
* ``em``    three EM iterations of lpmethods.em

A program builds the operator of a scan geometry once and passes every new batch of slices through it, so ``prepare``
keeps the last geometry's operator and makes new inputs: ellipse phantoms, or their sinograms with noise.
``exact`` evaluates the same operators in float64 with plain torch, from the formulas and the float32 tables' values.
"""
import math

import numpy as np
import torch

from lprec_amd import lpTransform, lpmethods
from lprec_amd.autograd import backprojection, radon

EM_ITERATIONS, EM_EPS = 3, 1e-3


def _case(name, op, n0, nproj, slices, cor=None, filt="none", interp="cubic"):
    case = {"op": op, "n0": n0, "nproj": nproj, "slices": slices, "cor": n0 / 2 if cor is None else cor,
            "filter": filt, "interp": interp}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # the smallest grid in use: a call is all latency and launches
        _case("fwd_64x1", "fwd", 64, 48, 1),
        # filtered back-projection of a few binned slices, as in a quick look during a scan
        _case("fbp_256x4", "adj", 256, 384, 4, filt="parzen"),
        # an odd detector width and angle count with the rotation centre off the middle, linear interpolation
        _case("fbp_501x5_linear", "adj", 501, 353, 5, cor=253.4, filt="ramp", interp="linear"),
        # a few iterations of a reconstruction method on a small stack: every pass runs fwd and adj
        _case("em_512x8", "em", 512, 384, 8),
        # gradient through the filtered back-projection with a centre offset (padded to 528)
        _case("bproj_512x8", "bproj", 512, 384, 8, cor=253.0, filt="parzen"),
        # projections of a medium stack whose centre offset pads the grid to 1056
        _case("fwd_1000x7", "fwd", 1000, 901, 7, cor=521.0),
        # one step of a gradient method on a medium stack through the differentiable operator
        _case("radon_1024x16", "radon", 1024, 1024, 16),
        # one full-size slice, off-centre (padded to 2064): looking for the rotation centre, slice by slice
        _case("fbp_2048x1", "adj", 2048, 1500, 1, cor=1024.912, filt="parzen"),
        # one slice of the widest detector
        _case("fwd_4096x1", "fwd", 4096, 1500, 1),
        # whole batches at full size: the two operators of every iterative method ...
        _case("fwd_2048x32", "fwd", 2048, 1500, 32),
        _case("adj_2048x32", "adj", 2048, 1500, 32),
        # ... and a production reconstruction of a scan whose centre is off the middle (padded to 2064)
        _case("fbp_2048x32", "adj", 2048, 1500, 32, cor=1024.912, filt="parzen"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another geometry: any detector width, angle count and batch, half of the scans off-centre."""
    op = rng.choice(["fwd", "adj", "adj", "radon", "bproj"])
    n0 = _log_int(rng, 64, 2048)
    if rng.random() < 0.3:   # a common detector size
        n0 = rng.choice([64, 128, 256, 512, 1024, 2048])
    nproj = max(48, min(2048, int(n0 * rng.uniform(0.5, 1.5))))
    most = 32 * 2048 * 2048 // (n0 * n0)
    slices = _log_int(rng, 1, max(1, min(32, most // (4 if op in ("radon", "bproj") else 1))))
    cor = n0 / 2 if rng.random() < 0.5 else round(n0 / 2 + n0 * rng.uniform(-0.02, 0.02), 2)
    filt = rng.choice(["ramp", "parzen", "shepp-logan", "hamming"]) if op in ("adj", "bproj") and rng.random() < 0.7 else "none"
    return _case(None, op, n0, nproj, slices, cor, filt, "linear" if rng.random() < 0.2 else "cubic")


def _needs_fwd(case):
    return case["op"] not in ("adj", "bproj")


def _ellipses(case, seed):
    """Per slice 12 ellipses inside the unit disk: value, half axes, centre, rotation."""
    g = torch.Generator().manual_seed(1000003 * int(seed) + 17)
    u = torch.rand((case["slices"], 12, 6), generator=g, dtype=torch.float64)
    val = 0.1 + 0.9 * u[..., 0]
    a, b = 0.05 + 0.25 * u[..., 1], 0.05 + 0.25 * u[..., 2]
    rad, ang = 0.6 * u[..., 3].sqrt(), 2 * math.pi * u[..., 4]
    return val, a, b, rad * ang.cos(), rad * ang.sin(), math.pi * u[..., 5]


def _images(case, seed):
    n = case["n0"]
    x = torch.linspace(-1, 1, n, device="cuda")[None, :]
    y = torch.linspace(-1, 1, n, device="cuda")[:, None]
    f = torch.zeros((case["slices"], n, n), device="cuda")
    pars = torch.stack(_ellipses(case, seed), -1).tolist()
    for s, rows in enumerate(pars):
        for val, a, b, x0, y0, psi in rows:
            c, d = math.cos(psi), math.sin(psi)
            u, v = (x - x0) * c + (y - y0) * d, (y - y0) * c - (x - x0) * d
            f[s].add_(((u / a) ** 2 + (v / b) ** 2 <= 1), alpha=val)
    return f


def _sinograms(case, seed):
    n, p = case["n0"], case["nproj"]
    th = (torch.arange(p, device="cuda") * (math.pi / p))[:, None]
    s = (2.0 * (torch.arange(n, device="cuda") - case["cor"]) / n)[None, :]
    R = torch.zeros((case["slices"], p, n), device="cuda")
    pars = torch.stack(_ellipses(case, seed), -1).tolist()
    for k, rows in enumerate(pars):
        for val, a, b, x0, y0, psi in rows:
            r2 = (a * torch.cos(th - psi)) ** 2 + (b * torch.sin(th - psi)) ** 2
            t = s - (x0 * torch.cos(th) + y0 * torch.sin(th))
            R[k].add_((r2 - t * t).clamp_min(0).sqrt() / r2, alpha=2 * val * a * b)
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 5)
    noise = torch.rand(R.shape, generator=g, device="cuda")
    return R.mul_(1 + 0.02 * noise).add_(noise, alpha=0.01)


_kept = {}


def _operator(case):
    key = tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "op"))) + (_needs_fwd(case),)
    if key not in _kept:
        for lp in _kept.values():
            torch.cuda.synchronize()
            lp.close()
        _kept.clear()
        lp = lpTransform(case["n0"], case["nproj"], case["slices"], case["filter"], case["cor"], case["interp"])
        lp.precompute(_needs_fwd(case))
        lp.initcmem(_needs_fwd(case), 0)
        _kept[key] = lp
    return _kept[key]


def prepare(case, seed):
    op, n, p, ns = case["op"], case["n0"], case["nproj"], case["slices"]
    state = {"op": op, "lp": _operator(case)}
    if op in ("fwd", "radon"):
        state["f"] = _images(case, seed)
    if op != "fwd":
        state["R"] = _sinograms(case, seed)
    if op == "fwd":
        state["out"] = torch.empty((ns, p, n), device="cuda")
    elif op == "adj":
        state["out"] = torch.empty((ns, n, n), device="cuda")
    elif op == "em":
        state["init"] = torch.full((ns, n, n), 1e-3, device="cuda")
    elif op == "radon":
        state["f"].requires_grad_(True)
    else:
        state["R"].requires_grad_(True)
        state["target"] = _images(case, seed)
    return state


def run(state):
    op, lp = state["op"], state["lp"]
    if op == "fwd":
        lp.fwdp(state["out"], state["f"], 0)
        return state["out"]
    if op == "adj":
        lp.adjp(state["out"], state["R"], 0)
        return state["out"]
    if op == "em":
        return lpmethods.em(lp, state["init"], state["R"], EM_ITERATIONS, EM_EPS, 0)
    if op == "radon":
        x, target, y = state["f"], state["R"], radon(state["f"], lp)
    else:
        x, target, y = state["R"], state["target"], backprojection(state["R"], lp)
    r = y - target
    (grad,) = torch.autograd.grad((r * r).sum(), x)
    return {"value": y.detach(), "gradient": grad}


def _padded(case):
    return int(math.ceil((case["n0"] + abs(case["n0"] / 2 - case["cor"]) * 2.0) / 16.0) * 16)


def work(case):
    """Bytes: inputs read and outputs written once (each operator of a call reads its input and writes its output).
    Flops: the transforms of the three 2N x N grids there and back (5 n log2 n per complex point, half of that for
    real data), the product with the kernel, and the 16-tap (4-tap) samples and the filter's transforms."""
    n0, p0, ns, n = case["n0"], case["nproj"], case["slices"], _padded(case)
    calls = {"fwd": 1, "adj": 1, "radon": 2, "bproj": 2, "em": 2 * EM_ITERATIONS + 1}[case["op"]]
    grid = 2.0 * n * n
    conv = 3 * (2 * 2.5 * grid * math.log2(grid) + 3 * grid)
    tap = 2 * 16 if case["interp"] == "cubic" else 2 * 4
    samples = tap * (3 * 0.3 * grid + (n0 * p0 if _needs_fwd(case) else 3 * 0.8 * n0 * n0))
    filt = p0 * 2 * 2.5 * 2 * n * math.log2(2 * n) if case["filter"] != "none" else 0.0
    return {"bytes": calls * ns * 4.0 * (n0 * n0 + n0 * p0), "flops": calls * ns * (conv + samples + filt)}


# ---- the same operators in float64 ----------------------------------------------------------------------------

BETA = math.pi / 3
AR = math.sin(BETA / 2) / (1 + math.sin(BETA / 2))
AM = (math.cos(BETA / 2) - math.sin(BETA / 2)) / (1 + math.sin(BETA / 2))


def _dev(a):
    return torch.as_tensor(a, device="cuda" if torch.cuda.is_available() else "cpu")


def _f32(t):
    """The float32 value that a table holds, as float64."""
    return t.to(torch.float32).double()


def _end_corrected(n):
    h = np.ones(n)
    c = 1 + np.array([-216254335, 679543284, -1412947389, 2415881496, -3103579086, 2939942400, -2023224114,
                      984515304, -321455811, 63253516, -5675265]) / 958003200.0
    h[0] = 2 * (c[0] - 0.5)
    h[1:11] *= c[1:]
    h[-10:] *= c[:0:-1]
    return h


class _Exact:
    def __init__(self, case):
        n0, p0, cor = case["n0"], case["nproj"], case["cor"]
        n = _padded(case)
        os_ = int(max(round(3.0 * n / 2.0 / p0), 1))
        self.n0, self.p0, self.n, self.os, self.p = n0, p0, n, os_, os_ * p0
        self.nt, self.nr, self.lb, self.o = n, 2 * n, n // 2 - int(cor), n // 2 - n0 // 2
        self.cubic, self.filter = case["interp"] == "cubic", case["filter"]
        t = np.linspace(-np.pi / 2, np.pi / 2, 1000)
        w = AR * np.cos(t) + (1 - AR) + 1j * AR * np.sin(t)
        self.g = float(np.max(np.log(np.abs(w)) + np.log(np.cos(BETA / 2 - np.arctan2(w.imag, w.real)))))
        self.span = self.g - math.log(AM)
        self.th = (np.arange(-n / 2, n / 2) * np.float64(np.float32(2 * BETA / n))).astype(np.float32)
        self.rh = (np.arange(-2 * n, 0) * (self.span / (2 * n))).astype(np.float32)
        self.proj = np.arange(0, self.p) * np.pi / self.p - BETA / 2
        self.prefilter = {}

    def spline(self, length):
        """Samples to cubic B-spline coefficients of a line, as a matrix."""
        if length not in self.prefilter:
            z = math.sqrt(3.0) - 2.0
            lam = (1 - z) * (1 - 1 / z)
            c = np.eye(length)
            first = c[0].copy()
            for k in range(min(12, length)):
                first += z ** (k + 1) * c[k]
            c[0] = lam * first
            for k in range(1, length):
                c[k] = lam * c[k] + z * c[k - 1]
            c[-1] *= z / (z - 1)
            for k in range(length - 2, -1, -1):
                c[k] = z * (c[k + 1] - c[k])
            self.prefilter[length] = _dev(c)
        return self.prefilter[length]

    def smooth(self, a):
        return self.spline(a.shape[0]) @ a @ self.spline(a.shape[1]).T if self.cubic else a

    def sample(self, grid, x, y):
        h, w = grid.shape
        flat, ix, iy = grid.reshape(-1), x.floor(), y.floor()
        fx, fy, ix, iy = x - ix, y - iy, ix.long(), iy.long()
        if self.cubic:
            def weights(f):
                o = 1 - f
                return o ** 3 / 6, 2 / 3 - 0.5 * f * f * (2 - f), 2 / 3 - 0.5 * o * o * (2 - o), f ** 3 / 6
            wx, wy, first = weights(fx), weights(fy), -1
        else:
            wx, wy, first = (1 - fx, fx), (1 - fy, fy), 0
        out = 0.0
        for b in range(len(wy)):
            row = torch.remainder(iy + first + b, h) * w
            line = 0.0
            for a in range(len(wx)):
                line = line + wx[a] * flat[row + torch.remainder(ix + first + a, w)]
            out = out + wy[b] * line
        return out

    def kernel(self, adjoint):
        """Spectrum of the log-polar kernel [2n, n / 2 + 1], its float32 values."""
        nl, nt, nr = 4 * self.nt, self.nt, self.nr
        thl = np.arange(-nl / 2, nl / 2) / nl * (2 * BETA)
        h, logcos = _dev(_end_corrected(nl)), _dev(np.log(np.cos(thl)))
        k = _dev(np.arange(-nr / 2, nr / 2)) * (2 * math.pi / self.span)
        out = torch.zeros((nr, nt), dtype=torch.complex128, device=h.device)
        rows = max(1, (1 << 25) // nl)
        for r in range(0, nr, rows):
            kk = k[r:r + rows, None]
            e = torch.polar((logcos * (0 if adjoint else -1)).exp().expand(len(kk), nl), (kk if adjoint else -kk) * logcos)
            F = torch.fft.fftshift(torch.fft.fft(torch.fft.fftshift(h * e, dim=1), dim=1), dim=1)
            out[r:r + rows] = F[:, nl // 2 - nt // 2:nl // 2 + nt // 2]
        out *= thl[1] - thl[0]
        out[0], out[:, 0] = 0, 0
        out = torch.fft.fftshift(out)[:, :nt // 2 + 1]
        n, p = self.n, self.p
        if adjoint:
            out = out * ((n + 1) * (n - 1) / n ** 2 / 2 * math.sqrt(self.os * p / n / 2))
        else:
            out = out * (math.sqrt(n * self.os / p) * math.pi / 4 / AR / math.sqrt(2))
        if self.cubic:
            out = out / torch.outer(self.b3(self.rh), self.b3(self.th)[:nt // 2 + 1])
        return torch.complex(_f32(out.real.contiguous()), _f32(out.imag.contiguous()))

    def b3(self, lattice):
        """Spectrum of the cubic B-spline sampled on the float32 lattice (its rounding is part of the operator)."""
        x = lattice.astype(np.float64)
        c = (len(x) + 2) // 2 - 1
        d = np.abs(x - x[c]) / (x[1] - x[0])
        v = np.where(d < 1, (3 * d ** 3 - 6 * d ** 2 + 4) / 6, np.where(d < 2, (-d ** 3 + 6 * d ** 2 - 12 * d + 8) / 6, 0.0))
        v[np.abs(np.arange(len(x)) - c) > 2] = 0
        return _dev(np.fft.fft(np.fft.ifftshift(v)))

    def convolve(self, grid, fz):
        return torch.fft.irfft2(torch.fft.rfft2(grid) * fz, s=(self.nr, self.nt))

    def forward_tables(self):
        n, th, rh = self.n, _dev(self.th.astype(np.float64)), _dev(self.rh.astype(np.float64))
        z1, z2 = torch.outer(rh.exp(), th.cos()).reshape(-1), torch.outer(rh.exp(), th.sin()).reshape(-1)
        self.fz_f, self.erho = self.kernel(False), _f32(rh.exp())[:, None]
        self.img, self.pol = [], []
        t0, t1, r0, r1 = (float(v) for v in (self.th[0], self.th[-1], self.rh[0], self.rh[-1]))
        s = _dev(np.linspace(-1, 1, n))
        for k in range(3):
            phi = k * BETA + BETA / 2
            c1 = ((z1 - (1 - AR)) * math.cos(phi) - z2 * math.sin(phi)) / AR
            c2 = -((z1 - (1 - AR)) * math.sin(phi) + z2 * math.cos(phi)) / AR
            ids = torch.nonzero(c1 ** 2 + c2 ** 2 <= 1)[:, 0]
            self.img.append((ids, _f32((c1[ids] + 1) / 2 * (n - 1)), _f32((c2[ids] + 1) / 2 * (n - 1))))
            rows = np.where((self.proj >= k * BETA - BETA / 2) & (self.proj < k * BETA + BETA / 2))[0]
            rows = rows[rows % self.os == 0]
            t = _dev(self.proj[rows] - k * BETA)[:, None]
            rho = torch.log(s[None, :] * AR + (1 - AR) * t.cos())
            x = ((t - t0) / (t1 - t0) * (self.nt - 1)).expand(len(rows), n)
            self.pol.append((_dev(rows // self.os), _f32(x), _f32((rho - r0) / (r1 - r0) * (self.nr - 1))))

    def forward(self, f):
        """One slice: image [n0, n0] -> sinogram [p0, n0]."""
        n, n0, o = self.n, self.n0, self.o
        img = self.smooth(torch.nn.functional.pad(f, (o, n - n0 - o, o, n - n0 - o)))
        R = torch.zeros((self.p0, n), dtype=torch.float64, device=f.device)
        for (ids, x, y), (rows, px, py) in zip(self.img, self.pol):
            lp = torch.zeros(self.nr * self.nt, dtype=torch.float64, device=f.device).index_put((ids,), self.sample(img, x, y))
            conv = self.convolve(lp.reshape(self.nr, self.nt) * self.erho, self.fz_f)
            R = R.index_put((rows,), self.sample(conv, px.reshape(-1), py.reshape(-1)).reshape(px.shape))
        return R[:, self.lb:self.lb + n0]

    def window(self):
        """The FBP filter's centred response of length 4n, its float32 values."""
        ne, d = 4 * self.n, 0.5
        t = np.arange(0, ne / 2 + 1) / ne
        k = 12   # weights that integrate t times polynomials of degree < k, on overlapping windows of k samples
        s = np.linspace(1e-40, 1, k)
        inv = np.linalg.inv(np.exp(np.outer(np.arange(k), np.log(s))))
        powers = np.arange(1, k + 2)
        u = np.diff(np.exp(np.outer(powers, np.log(s))) / powers[:, None])
        w1, w2 = inv @ u[1:], inv @ u[:-1]
        m = len(t)
        p = 1 / np.concatenate((np.arange(1, k), (k - 1) * np.ones(m - 2 * (k - 1) - 1), np.arange(k - 1, 0, -1)))
        j = np.arange(m - k + 1)
        a, pm = t[j + k - 1] - t[j], p[j[:, None] + np.arange(k - 1)]
        c = (a ** 2)[:, None] * (pm @ w1.T) + (a * t[j])[:, None] * (pm @ w2.T)
        w = np.zeros(m)
        for i in range(k):
            w[i:i + len(j)] += c[:, i]
        tail = w[-40] / (m - 40) * np.arange(m - 40, m)
        w[-40:] = tail
        w *= ne * 0.5
        w *= {"ramp": lambda: 1.0, "shepp-logan": lambda: np.sinc(t / (2 * d)) * (t / d <= 2),
              "cosine": lambda: np.cos(np.pi * t / (2 * d)) * (t / d <= 1),
              "cosine2": lambda: np.cos(np.pi * t / (2 * d)) ** 2 * (t / d <= 1),
              "hamming": lambda: (0.54 + 0.46 * np.cos(np.pi * t / d)) * (t / d <= 1),
              "hann": lambda: (1 + np.cos(np.pi * t / d)) / 2 * (t / d <= 1),
              "parzen": lambda: (1 - t / d) ** 3 * (t / d <= 1)}[self.filter]()
        w = w * (w >= 0)
        return np.concatenate((w[:0:-1], [2 * w[0]], w[1:]))[:-1].astype(np.float32).astype(np.float64)

    def adjoint_tables(self):
        n = self.n
        self.fz_a = self.kernel(True)
        lin = _dev(np.linspace(-1, 1, n))
        x1, x2 = lin[None, :].expand(n, n).reshape(-1), -lin[:, None].expand(n, n).reshape(-1)
        self.pix = torch.nonzero(x1 * x1 + x2 * x2 <= 1)[:, 0]
        x1, x2 = x1[self.pix], x2[self.pix]
        th, rh = self.th.astype(np.float64), self.rh.astype(np.float64)
        t0, t1, r0, r1 = th[0], th[-1], rh[0], rh[-1]
        cols = np.where((self.th >= np.float32(-BETA / 2)) & (self.th < np.float32(BETA / 2)))[0]
        tc = _dev(th[cols])

        def points(rows, rho):
            """Log-polar points of these rows, taken at rho: their index, column number and detector coordinate."""
            z = (_dev(np.exp(rho))[:, None] - (1 - AR) * tc.cos()[None, :]) / AR
            r, c = torch.nonzero(z.abs() <= 1, as_tuple=True)
            return _dev(rows)[r] * self.nt + _dev(cols)[c], c, _f32((z[r, c] + 1) / 2 * (n - 1))

        lz = np.log(np.exp(rh))
        up, down = np.where(lz > self.g)[0], np.where(lz < math.log(AM) - self.g + (rh[1] - rh[0]))[0]
        sets = [points(np.arange(self.nr), rh), points(up, lz[up] + math.log(AM) - self.g),
                points(down, lz[down] - math.log(AM) + self.g)]
        member = [np.where((self.proj >= k * BETA - BETA / 2) & (self.proj < k * BETA + BETA / 2))[0] for k in range(3)]
        first = [self.proj[m[0]] for m in member]
        last = [self.proj[m[-1]] - self.proj[m[0]] for m in member]
        per = (self.p - 1) / (first[2] + last[2] - first[0])
        self.sino, self.cart = [], []
        for k in range(3):
            angle = (tc + k * BETA - first[k]) / last[k] * (len(member[k]) - 1) + (first[k] - first[0]) * per
            self.sino.append([(ids, x, _f32(angle)[c]) for ids, c, x in sets])
            phi = k * BETA + BETA / 2
            z1 = AR * (x1 * math.cos(phi) + x2 * math.sin(phi)) + (1 - AR)
            z2 = AR * (-x1 * math.sin(phi) + x2 * math.cos(phi))
            self.cart.append((_f32((torch.atan2(z2, z1) - t0) / (t1 - t0) * (self.nt - 1)),
                              _f32((torch.log(torch.sqrt(z1 ** 2 + z2 ** 2)) - r0) / (r1 - r0) * (self.nr - 1))))
        if self.filter != "none":
            self.response = torch.fft.ifftshift(_dev(self.window()))

    def adjoint(self, R):
        """One slice: sinogram [p0, n0] -> image [n0, n0]."""
        n, n0, lb = self.n, self.n0, self.lb
        rows = torch.nn.functional.pad(R[None], (lb, n - n0 - lb), mode="replicate")[0]
        if self.filter != "none":
            rows = torch.fft.ifft(torch.fft.fft(rows, n=4 * n) * self.response).real[:, :n]
        at = torch.arange(self.p0, device=R.device) * self.os
        full = torch.zeros((self.p, n), dtype=torch.float64, device=R.device).index_put((at,), rows)
        full = self.smooth(full)
        img = torch.zeros(len(self.pix), dtype=torch.float64, device=R.device)
        for sets, (cx, cy) in zip(self.sino, self.cart):
            lp = torch.zeros(self.nr * self.nt, dtype=torch.float64, device=R.device)
            for ids, x, y in sets:
                if len(ids):
                    lp = lp.index_add(0, ids, self.sample(full, x, y))
            img = img + self.sample(self.convolve(lp.reshape(self.nr, self.nt), self.fz_a), cx, cy)
        full = torch.zeros(n * n, dtype=torch.float64, device=R.device).index_put((self.pix,), img)
        return full.reshape(n, n)[self.o:self.o + n0, self.o:self.o + n0]


def exact(case, seed):
    op, e = case["op"], _Exact(case)
    if op in ("fwd", "radon", "em"):
        e.forward_tables()
    if op in ("adj", "bproj", "em"):
        e.adjoint_tables()
    f = _images(case, seed).double() if op in ("fwd", "radon", "bproj") else None
    R = _sinograms(case, seed).double() if op != "fwd" else None
    if op == "fwd":
        return torch.stack([e.forward(v) for v in f])
    if op == "adj":
        return torch.stack([e.adjoint(v) for v in R])
    if op == "em":
        out, eps = [], float(np.float32(EM_EPS))
        for tomo in R:
            x = torch.full((e.n0, e.n0), float(np.float32(1e-3)), dtype=torch.float64, device=tomo.device)
            norm = e.adjoint(torch.ones_like(tomo)) + 1e-5
            for _ in range(EM_ITERATIONS):
                x = x * (e.adjoint(tomo / (e.forward(x) + eps)) / norm)
            out.append(x)
        return torch.stack(out)
    value, grads = [], []
    for v, target in zip(*((f, R) if op == "radon" else (R, f))):
        v.requires_grad_(True)
        y = e.forward(v) if op == "radon" else e.adjoint(v)
        r = y - target
        grads.append(torch.autograd.grad((r * r).sum(), v)[0])
        value.append(y.detach())
    return {"value": torch.stack(value), "gradient": torch.stack(grads)}
