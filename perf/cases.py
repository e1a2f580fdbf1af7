"""The workloads by which this framework's speed is judged.

A case is a dict of plain values; `kind` names the entry point and the rest
its sizes and observer.  `prepare` makes what a user's program holds before
the call (screens on the GPU, preallocated outputs, a planned survey), `run`
is one pass through the public entry points, `work` the bytes and operations
the pass cannot do without, `exact` the same outputs in plain numpy: the
radial and polar motion from the Weierstrass-Biermann formula (one formula
for every root configuration) and the integrals by Gauss-Legendre quadrature
along it, so nothing of the kernels' formulas is shared.
"""

import math

import numpy as np
import torch

import kgeo_amd.models as models
from kgeo_amd import batch, counts, equatorial, images, lensing, raytrace

R_O = 1.0e4


def _ray(name, na, nb, ngeo, a, inc, window, lean=False):
    return dict(name=name, kind="rays", na=na, nb=nb, ngeo=ngeo, a=a, inc=inc, window=window, lean=lean)


def listed():
    return [
        # raytrace_ana with the reference's own defaults: a line of 1000
        # pixels at beta = 0, 250 samples; the smallest call, latency-bound
        _ray("line_1000x250", 1000, 1, 250, 0.94, 20.0, 6.0),
        # a preview image, every output (tau, t, r, theta, phi, sigma)
        _ray("image_64sq_x100", 64, 64, 100, 0.94, 17.0, 8.0),
        # an odd-sized, nearly edge-on retrograde image, every output
        _ray("image_217x301_x333", 217, 301, 333, -0.9, 80.0, 10.0),
        # the headline image in a program that keeps its buffers and needs t, r, theta, phi
        _ray("image_512sq_x500", 512, 512, 500, 0.94, 17.0, 8.0, lean=True),
        # the drop-in call with numpy arrays in and out
        dict(name="dropin_100x90_x200", kind="dropin", na=100, nb=90, ngeo=200, a=0.7, inc=60.0, window=9.0),
        # coordinates at a few Mino times of the caller's (crossings, jet models)
        dict(name="points_150x140_x12", kind="points", na=150, nb=140, ngeo=12, a=0.8, inc=50.0, window=10.0),
        # a parameter survey of images of several sizes, planned once and replayed
        dict(name="survey_16", kind="survey", n=16),
        # the equatorial image with all its parts
        dict(name="equatorial_1024sq", kind="disk", na=1024, nb=1024, a=0.94, inc=17.0, window=12.0, mbar=2),
        # one gradient step's image and its derivative in (a, theta_o, p)
        dict(name="gradient_256sq", kind="gradient", na=256, nb=256, a=0.7, inc=40.0, window=12.0, mbar=2),
        # the polarized image with two subrings
        dict(name="polarized_800sq", kind="polarized", na=800, nb=800, a=0.7, inc=45.0, window=10.0, mbar=1),
        # lensed curves of the horizon for a few observers, subrings 0..5
        dict(name="curves_24x6x360", kind="curves", n=24, nphi=360),
        # crossing and turning counts along sampled rays
        dict(name="counts_256sq_x100", kind="counts", na=256, nb=256, ngeo=100, a=0.6, inc=70.0, window=8.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rays", "rays", "rays", "rays", "survey", "dropin", "points", "disk", "gradient", "polarized",
                       "curves", "counts"])
    a = round(rng.choice([-1.0, 1.0, 1.0]) * rng.uniform(0.05, 0.98), 3)
    inc = round(rng.choice([rng.uniform(5.0, 85.0), rng.uniform(5.0, 85.0), rng.uniform(95.0, 165.0)]), 1)
    window = round(rng.uniform(6.0, 12.0), 2)

    def side(lo, hi):
        n = _log(rng, lo, hi)
        return n, max(1, int(n * rng.uniform(0.6, 1.0)))

    if kind == "survey":
        return dict(kind=kind, n=rng.randint(4, 16))
    if kind == "curves":
        return dict(kind=kind, n=rng.randint(2, 24), nphi=rng.randint(60, 360))
    if kind in ("disk", "gradient", "polarized"):
        lo, hi, mb = {"disk": (96, 1024, (0, 2)), "gradient": (64, 256, (1, 2)), "polarized": (90, 800, (0, 1))}[kind]
        na, nb = side(lo, hi)
        return dict(kind=kind, na=na, nb=nb, a=a, inc=inc, window=window, mbar=rng.randint(*mb))
    if kind == "points":
        na, nb = side(24, 150)
        return dict(kind=kind, na=na, nb=nb, ngeo=rng.randint(1, 12), a=a, inc=inc, window=window)
    if kind == "counts":
        na, nb = side(40, 256)
        return dict(kind=kind, na=na, nb=nb, ngeo=rng.randint(10, 100), a=a, inc=min(inc, 180.0 - inc), window=window)
    if kind == "dropin":
        na, nb = side(30, 100)
        return dict(kind=kind, na=na, nb=nb, ngeo=rng.randint(50, 200), a=a, inc=inc, window=window)
    na, nb = side(32, 512)
    return dict(kind=kind, na=na, nb=nb, ngeo=_log(rng, 50, 500), a=a, inc=inc, window=window,
                lean=rng.random() < 0.5)


def _observer(case, seed):
    """The case's spin and inclination moved a little by the seed, and its
    screen moved by a fraction of a pixel, so that another seed is another image."""
    rng = np.random.default_rng(seed)
    a = float(np.clip(case["a"] + rng.uniform(-0.02, 0.02), -0.99, 0.99))
    if abs(a) < 0.02:
        a = 0.02
    th = float((case["inc"] + rng.uniform(-2.0, 2.0)) * np.pi / 180.0)
    w, na, nb = case["window"], case["na"], case["nb"]
    al = np.linspace(-w, w, na) + rng.uniform(-0.5, 0.5) * 2.0 * w / na
    be = np.linspace(-w, w, nb) + rng.uniform(-0.5, 0.5) * 2.0 * w / nb if nb > 1 else np.zeros(1)
    A, B = np.meshgrid(al, be)
    return a, th, A.flatten(), B.flatten(), rng


def _survey_images(case, seed):
    """Spins and inclinations as batch.survey_draw has them; resolutions and
    sample counts run through their range, so that every seed is as much work."""
    d = batch.survey_draw(case["n"], seed)
    rng = np.random.default_rng([seed, 1])
    for k, im in enumerate(d):
        im["res"] = (64, 128, 256, 512)[k % 4]
        im["ngeo"] = 50 + (k * 147) % 351
    shift = rng.uniform(-0.01, 0.01, (case["n"], 2))
    out = batch.survey_images(d)
    for im, s in zip(out, shift):
        im["alpha"] = im["alpha"] + s[0]
        im["beta"] = im["beta"] + s[1]
    return out


def _models():
    return dict(emissivity=models.Emissivity("ring"),
                velocity=models.Velocity("general", fac_subkep=0.6, beta_r=0.7, beta_phi=0.8),
                bfield=models.Bfield("bz_guess", C=1.0))


def _taus(a, th, A, B, n, rng, tau_tot):
    """Mino times of the caller's: sorted along each ray, inside its range."""
    u = np.sort(rng.uniform(0.02, 0.98, (n, len(A))), axis=0)
    return u * tau_tot[None, :]


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "survey":
        s["survey"] = batch.BatchSurvey(_survey_images(case, seed), tuning=(128, 16))
        return s
    if kind == "curves":
        rng = np.random.default_rng(seed)
        spins = np.repeat(rng.uniform(0.01, 0.99, case["n"]), 6)
        s.update(spins=spins, incs=np.repeat(rng.uniform(1.0, 89.0, case["n"]) * np.pi / 180.0, 6),
                 reqs=1.0 + np.sqrt(1.0 - spins ** 2), mbars=np.tile(np.arange(6, dtype=np.int32), case["n"]),
                 varphis=np.linspace(-180.0, 179.0, case["nphi"]) * np.pi / 180.0)
        return s
    a, th, A, B, rng = _observer(case, seed)
    s.update(a=a, th=th, A=A, B=B)
    if kind == "dropin":
        return s
    dev = torch.device("cuda")
    s["alpha"], s["beta"] = torch.from_numpy(A).to(dev), torch.from_numpy(B).to(dev)
    if kind == "rays" and case["lean"]:
        n = len(A)
        s["out"] = {k: torch.empty((case["ngeo"], n), device=dev, dtype=torch.float64) for k in ("t", "r", "th", "ph")}
    if kind in ("points", "counts"):
        s["tau"] = torch.from_numpy(_taus(a, th, A, B, case["ngeo"], rng, _mino_total(a, th, A, B))).to(dev)
    if kind == "gradient":
        s["theta"] = torch.tensor([a, th, 2.0], dtype=torch.float64, device=dev, requires_grad=True)
        s["target"] = torch.from_numpy(rng.uniform(0.0, 0.05, len(A))).to(dev)
    if kind == "polarized":
        s["models"] = _models()
    return s


LABELS = ("rclass", "thclass", "nmax_eq", "tau_tot", "status")


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "rays":
        want = ("t", "r", "th", "ph") if case["lean"] else ("tau", "t", "r", "th", "ph", "sig")
        res = raytrace.raytrace_ana_device(s["a"], R_O, s["th"], s["alpha"], s["beta"], case["ngeo"], want=want,
                                           out=s.get("out"))
        return {k: getattr(res, k) for k in want + LABELS}
    if kind == "dropin":
        g = raytrace.raytrace_ana(a=s["a"], observer_coords=[0, R_O, s["th"], 0], image_coords=[s["A"], s["B"]],
                                  ngeo=case["ngeo"], plotdata=False)
        t, r, th, ph = g.geo_coords
        return dict(tau=g.mino_times, sig=g.affine_times, t=t, r=r, th=th, ph=ph)
    if kind == "points":
        sig, (t, r, th, ph) = raytrace.coords_at_tau_device(s["a"], R_O, s["th"], s["alpha"], s["beta"], s["tau"])
        return dict(sig=sig, t=t, r=r, th=th, ph=ph)
    if kind == "survey":
        sv = s["survey"]
        sv.run()
        return dict(sv.arena, **{k: getattr(sv, k) for k in LABELS})
    if kind == "disk":
        return equatorial.equatorial_image_device(s["a"], R_O, s["th"], s["alpha"], s["beta"], case["mbar"], 2.0)
    if kind == "gradient":
        s["theta"].grad = None
        img = equatorial.EquatorialImageFn.apply(s["theta"], s["alpha"], s["beta"], R_O, case["mbar"])
        torch.sum((img - s["target"]) ** 2).backward()
        return dict(image=img.detach(), grad=s["theta"].grad)
    if kind == "polarized":
        out = images.stokes_device(s["a"], np.inf, s["th"], case["mbar"], s["alpha"], s["beta"], polarization=True,
                                   specind=1.0, **s["models"])
        return {k: v for k, v in out.items() if isinstance(v, torch.Tensor)}
    if kind == "curves":
        rho, status = lensing.rho_of_req_device(s["spins"], s["incs"], s["reqs"], s["mbars"], s["varphis"])
        return dict(rho=rho, status=status)
    n_eq, n_pol = counts.crossings_device(s["a"], s["th"], s["alpha"], s["beta"], s["tau"])
    return dict(n_eq=n_eq, n_pol=n_pol,
                **counts.turnings_device(s["a"], s["th"], s["alpha"], s["beta"], s["tau"]))


# Operations the paths cannot do without, by the cheapest forms known here:
# a closed-form sample of one coordinate set is about 100 multiply-adds, a
# pixel's roots, labels and complete integrals about 2,000 operations, one
# direct elliptic evaluation of all five integrals about 3,000.
SAMPLE, PIXEL, POINT = 200.0, 2000.0, 3000.0


def work(case):
    kind = case["kind"]
    if kind == "survey":
        ims = [((64, 128, 256, 512)[k % 4] ** 2, 50 + (k * 147) % 351) for k in range(case["n"])]
        pix, smp = sum(p for p, _ in ims), sum(p * g for p, g in ims)
        return dict(bytes=16.0 * pix + 32.0 * smp + 18.0 * pix, flops=PIXEL * pix + SAMPLE * smp)
    if kind == "curves":
        roots = 6.0 * case["n"] * case["nphi"]
        return dict(bytes=12.0 * roots, flops=8.0 * PIXEL * roots)
    pix = float(case["na"] * case["nb"])
    if kind in ("rays", "dropin"):
        smp = pix * case["ngeo"]
        outs = 4 if case.get("lean") else 6
        return dict(bytes=34.0 * pix + 8.0 * outs * smp, flops=PIXEL * pix + SAMPLE * smp)
    if kind == "points":
        smp = pix * case["ngeo"]
        return dict(bytes=16.0 * pix + 48.0 * smp, flops=PIXEL * pix + POINT * smp)
    if kind == "counts":
        smp = pix * case["ngeo"]
        return dict(bytes=16.0 * pix + 37.0 * smp, flops=PIXEL * pix + 30.0 * smp)
    sub = case["mbar"] + 1
    if kind == "disk":
        return dict(bytes=pix * (16.0 + 21.0 + 32.0 * sub), flops=pix * (PIXEL + 300.0 * sub))
    if kind == "gradient":
        return dict(bytes=pix * 40.0, flops=4.0 * pix * (PIXEL + 300.0 * sub))
    return dict(bytes=pix * (32.0 + 56.0 * sub), flops=pix * (PIXEL + 1000.0 * sub))


# ---------------------------------------------------------------------------
# The outputs in plain numpy
# ---------------------------------------------------------------------------
def _rf(x, y, z):
    """Carlson R_F (real or complex) by duplication."""
    x, y, z = (np.asarray(v) + 0j for v in (x, y, z))
    for _ in range(26):
        lam = np.sqrt(x) * np.sqrt(y) + np.sqrt(y) * np.sqrt(z) + np.sqrt(z) * np.sqrt(x)
        x, y, z = (x + lam) / 4, (y + lam) / 4, (z + lam) / 4
    return 1.0 / np.sqrt((x + y + z) / 3.0)


def _jacobi(u, m):
    """sn, cn, dn for 0 <= m < 1 by the arithmetic-geometric mean."""
    a, b, c = np.ones_like(m), np.sqrt(1.0 - m), np.sqrt(m)
    ratio = []
    for _ in range(7):
        a, b, c = (a + b) / 2, np.sqrt(a * b), (a - b) / 2
        ratio.append(c / a)
    phi = 2.0 ** len(ratio) * a * u
    for q in reversed(ratio):
        phi = (phi + np.arcsin(q * np.sin(phi))) / 2
    sn, cn = np.sin(phi), np.cos(phi)
    return sn, cn, np.sqrt(1.0 - m * sn * sn)


class _Motion:
    """x(tau) of (dx/dtau)^2 = f(x) = sum f[k] x^k, x(0) = x0, dx/dtau(0) = v0."""

    def __init__(self, f, x0, v0):
        f0, f1, f2, f3, f4 = (np.asarray(c, float) + 0.0 * v0 for c in f)
        self.f, self.x0, self.v0 = (f0, f1, f2, f3, f4), x0, v0
        self.g2 = f4 * f0 - f3 * f1 / 4 + f2 * f2 / 12
        self.g3 = f4 * f2 * f0 / 6 + f3 * f2 * f1 / 48 - f2 ** 3 / 216 - f4 * f1 * f1 / 16 - f3 * f3 * f0 / 16
        comp = np.zeros(self.g2.shape + (3, 3))
        comp[..., 1, 0] = comp[..., 2, 1] = 1.0
        comp[..., 0, 2], comp[..., 1, 2] = self.g3 / 4, self.g2 / 4
        e = np.linalg.eigvals(comp).astype(complex)
        self.three = self.g2 ** 3 - 27 * self.g3 ** 2 > 0
        real = np.sort(e.real, axis=-1)
        single = np.take_along_axis(e, np.argmin(np.abs(e.imag), axis=-1)[..., None], -1)[..., 0].real
        self.e1 = np.where(self.three, real[..., 2], single)
        other = np.sqrt((self.g2 - 3.0 * self.e1 ** 2) / 4 + 0j)  # e2, e3 = -e1/2 +- ...
        self.e2, self.e3 = -self.e1 / 2 + other, -self.e1 / 2 - other
        self.d = (f0 + x0 * (f1 + x0 * (f2 + x0 * (f3 + x0 * f4))), f1 + x0 * (2 * f2 + x0 * (3 * f3 + x0 * 4 * f4)),
                  2 * f2 + x0 * (6 * f3 + x0 * 12 * f4), 6 * f3 + 24 * f4 * x0, 24 * f4)

    def at(self, tau):
        three = self.three
        h = np.sqrt(np.abs(3 * self.e1 ** 2 - self.g2 / 4))
        scale = np.where(three, np.sqrt(np.abs(self.e1 - self.e3.real)), 2 * np.sqrt(h))
        m = np.where(three, (self.e2.real - self.e3.real) / (self.e1 - self.e3.real), 0.5 - 0.75 * self.e1 / h)
        sn, cn, dn = _jacobi(scale * tau, np.clip(m, 0.0, 1.0 - 1e-16))
        s2 = sn * sn
        cot = np.where(cn > 0, (1 + cn) ** 2 / s2, s2 / (1 - cn) ** 2)
        p = np.where(three, self.e3.real + scale ** 2 / s2, self.e1 + h * cot)
        q = np.where(three, -2 * scale ** 3 * cn * dn / (s2 * sn),
                     -4 * h * np.sqrt(h) * dn * np.where(cn > 0, (1 + cn) ** 2 / (s2 * sn), sn / (1 - cn) ** 2))
        f0, f1, f2, f3, f4 = self.d
        b = p - f2 / 24
        moved = (-self.v0 * q + f1 * b / 2 + f0 * f3 / 24) / (2 * b * b - f0 * f4 / 48)
        return self.x0 + np.where(tau == 0.0, 0.0, moved)

    def time_to(self, x, turning):
        """The first tau at which the motion, moving straight there, is at x (a root of f where `turning`)."""
        f0, f1, f2 = self.d[:3]
        g0, g1, g2, g3, g4 = self.f
        fx = np.where(turning, 0.0, np.maximum(g0 + x * (g1 + x * (g2 + x * (g3 + x * g4))), 0.0))
        fpx = g1 + x * (2 * g2 + x * (3 * g3 + x * 4 * g4))
        dx = x - self.x0
        p = (np.sqrt(fx * f0) + f0) / (2 * dx * dx) + f1 / (4 * dx) + f2 / 24
        q = -(fx / dx ** 3 - fpx / (4 * dx * dx)) * np.sqrt(f0) - (f0 / dx ** 3 + f1 / (4 * dx * dx)) * np.sqrt(fx)
        z = _rf(p - self.e1, p - self.e2, p - self.e3).real
        half = _rf(0.0, self.e1 - self.e2, self.e1 - self.e3).real
        return np.where((q > 0) & ~turning, 2 * half - z, z)


class _Rays:
    def __init__(self, a, th, A, B):
        self.a, self.ap = a, np.asarray(A)
        self.lam = -A * np.sin(th)
        self.eta = (A * A - a * a) * np.cos(th) ** 2 + B * B
        al = a * a - self.eta - self.lam ** 2
        bl = 2.0 * (self.eta + (self.lam - a) ** 2)
        cl = -a * a * self.eta
        self.rp = 1.0 + math.sqrt(1.0 - a * a)
        w0 = 1.0 / R_O
        f = (np.ones_like(al), np.zeros_like(al), al, bl, cl)
        self.radial = _Motion(f, w0, np.sqrt(1.0 + w0 * w0 * (al + w0 * (bl + w0 * cl))))
        c0 = np.cos(th)
        big = self.eta + self.lam ** 2 - a * a
        v0 = np.sqrt(np.maximum(self.eta - c0 * c0 * (big + a * a * c0 * c0), 0.0))
        self.polar = _Motion((self.eta, 0.0 * al, -big, 0.0 * al, np.full_like(al, -a * a)), c0,
                             np.where(np.asarray(B) >= 0, 1.0, -1.0) * v0)
        # the largest root from the resolvent cubic, whose roots are the -e
        # (the invariants do not change under r = 1/w)
        z2 = -np.where(self.radial.three, self.radial.e3.real, self.radial.e1) - al / 6
        h2 = -al / 2 - z2 - bl / (4 * np.sqrt(z2))
        r4 = np.where(h2 >= 0, np.sqrt(z2) + np.sqrt(np.maximum(h2, 0)), -np.inf)
        self.turns = r4 > self.rp
        w1 = 1.0 / np.where(self.turns, r4, self.rp)
        for _ in range(3):  # the root of f again, by Newton
            fw, dfw = 1 + w1 * w1 * (al + w1 * (bl + w1 * cl)), w1 * (2 * al + w1 * (3 * bl + 4 * w1 * cl))
            w1 = np.where(self.turns & (np.abs(dfw) > 1e-6), w1 - fw / np.where(dfw == 0, 1.0, dfw), w1)
        t = self.radial.time_to(w1, self.turns)
        self.total = np.where(self.turns, 2 * t, t)

    def coords(self, tau):
        """(sig, t, r, th, ph) at Mino times tau [n][npix] that rise along each ray."""
        n, npix = tau.shape
        left = np.concatenate([[0.0], 1e-5 * 1.6 ** np.arange(24)])
        right = 1.0 - 1e-10 * 1.6 ** np.arange(49)
        x = np.concatenate([left, np.linspace(0.05, 0.95, 30), right])
        x = np.sort(x[(x >= 0) & (x < 1)])
        out = [np.empty_like(tau) for _ in range(5)]
        node, weight = np.polynomial.legendre.leggauss(8)
        for lo in range(0, npix, 256):
            sl = slice(lo, lo + 256)
            part = self._part(sl)
            ta = tau[:, sl]
            mesh = np.concatenate([x[:, None] * np.maximum(part.total, ta[-1]), ta])
            order = np.argsort(mesh, axis=0, kind="stable")
            mesh = np.take_along_axis(mesh, order, 0)
            place = np.argsort(order, axis=0, kind="stable")[len(x):]
            half = np.diff(mesh, axis=0) / 2
            at = mesh[:-1, None] + half[:, None] * (node[None, :, None] + 1.0)
            with np.errstate(all="ignore"):
                rates = part._rates(at)
                sums = []
                for v in rates:
                    inc = np.where(half > 0, half * np.sum(weight[None, :, None] * v, axis=1), 0.0)
                    sums.append(-np.take_along_axis(np.concatenate([0 * inc[:1], np.cumsum(inc, axis=0)]), place, 0))
                r, c = part._rc(ta)
            for o, v in zip(out, (sums[0], sums[1], r, np.arccos(np.clip(c, -1, 1)), sums[2])):
                o[:, sl] = v
        return out

    def _part(self, sl):
        p = object.__new__(_Rays)
        p.a, p.lam, p.total = self.a, self.lam[sl], self.total[sl]
        for k in ("radial", "polar"):
            m, src = object.__new__(_Motion), getattr(self, k)
            for name, v in src.__dict__.items():
                cut = lambda y: y[sl] if isinstance(y, np.ndarray) and y.ndim else y  # noqa: E731
                setattr(m, name, tuple(cut(y) for y in v) if isinstance(v, tuple) else cut(v))
            setattr(p, k, m)
        return p

    def _rc(self, tau):
        return 1.0 / self.radial.at(tau), self.polar.at(tau)

    def _rates(self, tau):
        r, c = self._rc(tau)
        a, lam = self.a, self.lam
        s2 = 1.0 - c * c
        delta = r * r - 2.0 * r + a * a
        return (r * r + a * a * c * c, (r * r + a * a) * (r * r + a * a - a * lam) / delta + a * (lam - a * s2),
                a * (2.0 * r - a * lam) / delta + lam / s2)


def _mino_total(a, th, A, B):
    with np.errstate(all="ignore"):
        return _Rays(a, th, A, B).total


def _turning_time(a, th, lam, eta):
    """K and F of the polar motion over its frequency's modulus, and the frequency, for eta > 0."""
    d = 0.5 * (1.0 - (eta + lam * lam) / (a * a))
    s = np.sqrt(d * d + eta / (a * a))
    up, um = d + s, d - s
    up = np.maximum(up, np.cos(th) ** 2)
    k, x = up / um, np.cos(th) / np.sqrt(up)
    return (_rf(0.0, 1.0 - k, 1.0).real, x * _rf(1.0 - x * x, 1.0 - k * x * x, 1.0).real, np.sqrt(-a * a * um))


def _exact_disk(a, th, A, B, mbar, p):
    rays = _Rays(a, th, A, B)
    lam, eta = rays.lam, rays.eta
    up = eta > 0
    K, F, w = _turning_time(a, th, lam, np.where(up, eta, 1.0))
    north, x = th < 0.5 * np.pi, rays.total * w
    flip = (B > 0) if north else (B < 0)  # the ray first moves away from the equator
    F0 = F if north else -F
    nmax = np.where(flip, np.floor((x + F0) / (2 * K)) - 1, np.floor((x - F0) / (2 * K)))
    sa, sp = np.sign(a), abs(a)
    z1 = 1 + np.cbrt(1 - a * a) * (np.cbrt(1 + a) + np.cbrt(1 - a))
    z2 = np.sqrt(3 * a * a + z1 * z1)
    ri = 3 + z2 - np.sqrt((3 - z1) * (3 + z1 + 2 * z2))
    out = {k: np.zeros((mbar + 1, len(A))) for k in ("I", "g", "r_s", "Ir")}
    for m in range(mbar + 1):
        msub = m + flip
        Ir = (2 * msub * K + np.where(flip, -F0, F0)) / w
        r = np.where(nmax >= m, 1.0 / rays.radial.at(np.maximum(Ir, 1e-13)), 0.0)
        lit = up & (nmax >= m) & (r > rays.rp)
        rr = np.where(lit, r, 2.0 * ri)
        r15, q = rr ** 1.5, rr - ri
        u0k = (r15 + sp) / np.sqrt(np.where(q >= 0, rr ** 3 - 3 * rr * rr + 2 * sp * r15, 1.0))
        delta, sri = rr * rr - 2 * rr + a * a, np.sqrt(ri)
        ell = sa * (ri * ri + a * a - 2 * sp * sri) / (ri ** 1.5 - 2 * sri + sp)
        gam, H = np.sqrt(1 - 2 / (3 * ri)), (2 * rr - a * ell) / delta
        u0 = np.where(q >= 0, u0k, gam * (1 + 2 / rr * (1 + H)))
        u1 = np.where(q >= 0, 0.0, -np.sqrt(2 / (3 * ri)) * np.maximum(ri / rr - 1, 0) ** 1.5)
        u3 = np.where(q >= 0, sa / (r15 + sp) * u0k, gam * (ell + a * H) / (rr * rr))
        R = (rr * rr + a * a - a * lam) ** 2 - delta * (eta + (lam - a) ** 2)
        kr = np.where(~rays.turns | (Ir <= 0.5 * rays.total), 1.0, -1.0)
        g = 1.0 / (u0 - lam * u3 - kr * u1 * np.sqrt(np.maximum(R, 0)) / delta)
        out["Ir"][m] = np.where(up, Ir, -1.0)
        out["r_s"][m] = np.where(up, r, -1.0)
        out["g"][m] = np.where(lit, g, 0.0)
        out["I"][m] = np.where(lit, g ** 3 * rr ** -p, 0.0)
    out["image"] = out["I"].sum(axis=0)
    out["Imax"] = np.where(up, rays.total, -1.0)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("rays", "dropin") and case["na"] * case["nb"] * (case["ngeo"] + 100) > 3_500_000:
        return None
    if kind in ("survey", "curves", "polarized", "counts"):
        return None
    a, th, A, B, rng = _observer(case, seed)
    with np.errstate(all="ignore"):
        if kind == "disk":
            out = _exact_disk(a, th, A, B, case["mbar"], 2.0)
            return dict(out, Nmax=None, zero_mask=None)
        if kind == "gradient":
            return dict(image=_exact_disk(a, th, A, B, case["mbar"], 2.0)["image"], grad=None)
        rays = _Rays(a, th, A, B)
        if kind == "points":
            tau = _taus(a, th, A, B, case["ngeo"], rng, rays.total)
            sig, t, r, thv, ph = rays.coords(tau)
            return dict(sig=sig, t=t, r=r, th=thv, ph=ph)
        stop = raytrace.MAXTAUFRAC * rays.total
        tau = np.linspace(0.0, stop, case["ngeo"])
        sig, t, r, thv, ph = rays.coords(tau)
        got = dict(tau=tau, t=t, r=r, th=thv, ph=ph, sig=sig)
        if kind == "dropin":
            return got
        if case["lean"]:
            got = {k: got[k] for k in ("t", "r", "th", "ph")}
        return dict(got, tau_tot=rays.total, **{k: None for k in LABELS if k != "tau_tot"})
