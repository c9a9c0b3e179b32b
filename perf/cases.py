"""Workloads by which the imaging path's speed is measured, through its public entry points.

Four kinds of work, each as a user's program calls it:

* ``image``:  lofar_amd.imager.image, samples to dirty image (grid, per-plane FFT, w-phase,
  plane sum), with the caller's scratch cube and image kept between calls;
* ``degrid``: lofar_amd.imager.degrid, the exact adjoint (sky image to model visibilities);
* ``fit``:    one chi^2 gradient evaluation of a sky model through torch.autograd
  (lofar_amd.autograd: planned degridding forward, planned imaging backward);
* ``dropin``: the reference's own call chain on host arrays, wstack() -> fftw_data()'s
  transform -> phase_correction().

Two samplings of the uv plane: ``disk`` (baselines uniform in a disk, in random order, the
synthetic observations of this repository's benchmark and tests) and ``tracks`` (an
interferometer with a dense core: Earth-rotation tracks in time order, so most samples fall
into the few tiles around the centre).  Visibilities are point and Gaussian sources plus
noise; ``flagged`` is the share of samples whose real part is NaN (skipped by the gridder).
"""
import math

import numpy as np
import torch

from lofar_amd import autograd, imager

PI_REF = 3.14159265359  # the reference's value (w-stacking.h:6)
DEV = "cuda"


def _case(name, kind, precision, n, nx, ny, nw, support, coverage="disk", F=1, P=1, flagged=0.0):
    return dict(name=name, kind=kind, precision=precision, n=n, nx=nx, ny=ny, nw=nw,
                support=support, coverage=coverage, F=F, P=P, flagged=flagged)


def listed():
    return [
        # a quick look at a small field: launches and latency count (the smoke size)
        _case("image_fp64_256", "image", "fp64", 20000, 256, 256, 4, 7),
        # a snapshot image in the fast mode
        _case("image_fp32c_1024", "image", "fp32c", 1 << 20, 1024, 1024, 8, 7),
        # the headline: a full-size FP64 image
        _case("image_fp64_4096", "image", "fp64", 1 << 24, 4096, 4096, 32, 7),
        # the same field from four times the samples in the fast mode
        _case("image_fp32c_4096", "image", "fp32c", 1 << 26, 4096, 4096, 32, 7),
        # a wide field: 8192-wide planes, the wider window of the streamed observations
        _case("image_fp32c_8192", "image", "fp32c", 1 << 25, 8192, 8192, 32, 9),
        # a side that is no power of two, as fftw_data() plans it, and a ragged sample count
        _case("image_fp64_3000", "image", "fp64", 2999999, 3000, 3000, 16, 7),
        # a core-dominated array's observation: channels and polarisations, flagged data
        _case("image_fp64_tracks", "image", "fp64", 1049505, 2048, 2048, 16, 7, "tracks", 4, 2,
              0.01),
        # model visibilities of a full-size sky image in the fast mode
        _case("degrid_fp32c_4096", "degrid", "fp32c", 1 << 24, 4096, 4096, 32, 7),
        # FP64 model visibilities along tracks on a field that is not square
        _case("degrid_fp64_tracks", "degrid", "fp64", 2999983, 2048, 1024, 12, 9, "tracks"),
        # calibration-style fitting, one gradient, FP64 at moderate size
        _case("fit_fp64_1024", "fit", "fp64", 1 << 20, 1024, 1024, 8, 7),
        # one iteration of the full-size sky-model fit in the fast mode
        _case("fit_fp32c_4096", "fit", "fp32c", 1 << 24, 4096, 4096, 32, 7),
        # an unchanged program of the reference: host arrays in and out
        _case("dropin_fp64_1024", "dropin", "fp64", 1 << 20, 1024, 1024, 8, 7),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("image", "image", "image", "degrid", "degrid", "fit", "dropin"))
    precision = "fp64" if kind == "dropin" else rng.choice(("fp64", "fp32c"))
    # sides that are no powers of two: FP64 images and drop-ins, degridding in both modes
    mixed = rng.random() < 0.35 and kind != "fit" and not (kind == "image" and
                                                           precision == "fp32c")
    sides = (300, 480, 720, 1000, 1250, 1536, 2000, 2400, 3000, 3600) if mixed else (
        256, 512, 1024, 2048, 4096)
    if kind == "dropin":
        sides = tuple(s for s in sides if s <= 1024)
    nx = rng.choice(sides)
    ny = nx if rng.random() < 0.6 else rng.choice(sides)
    nw = rng.randint(1, 8 if kind == "dropin" else 32)
    support = rng.choice((5, 7, 7, 7, 9, 9, 13))
    F, P = rng.choice(((1, 1), (1, 1), (2, 1), (1, 2), (4, 2))) if kind == "image" else (1, 1)
    # between a sparse and a well-filled cube of these planes
    top = min(1 << 24, 16 * nx * ny) // (F * P)
    n = _log_int(rng, max(2000, top // 2000), top) | 1
    coverage = rng.choice(("disk", "tracks"))
    flagged = 0.01 if kind in ("image", "dropin") and rng.random() < 0.5 else 0.0
    c = _case("", kind, precision, n, nx, ny, nw, support, coverage, F, P, flagged)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# inputs

def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + salt) % (1 << 62))
    return g


def _disk(n, g):
    """(u, v, w) of n baselines in units of the longest one's uv length."""
    f64 = dict(dtype=torch.float64, device=DEV)
    r = torch.sqrt(torch.rand(n, generator=g, **f64))
    th = 2 * math.pi * torch.rand(n, generator=g, **f64)
    w = torch.clamp(0.1 * torch.randn(n, generator=g, **f64), -0.3, 0.3)
    return r * torch.cos(th), r * torch.sin(th), w, 0.3


def _tracks(n, seed):
    """n samples, time-major, of an array of 62 stations: 24 in a core of 2 % of the array's
    extent, the others log-uniform out to it; declination 52 degrees, 8 hours."""
    rng = np.random.default_rng(seed)
    core, rest = 24, 38
    rad = np.concatenate([0.02 * np.sqrt(rng.random(core)),
                          np.exp(rng.uniform(math.log(0.02), 0.0, rest))])
    az = 2 * math.pi * rng.random(core + rest)
    east, north = rad * np.cos(az), rad * np.sin(az)
    lat, dec = math.radians(53.0), math.radians(52.0)
    xyz = np.stack([-math.sin(lat) * north, east, math.cos(lat) * north])
    i, j = np.triu_indices(core + rest, 1)
    b = xyz[:, j] - xyz[:, i]
    b /= np.sqrt((b ** 2).sum(0).max())
    f64 = dict(dtype=torch.float64, device=DEV)
    bx, by, bz = (torch.tensor(x, **f64).view(1, -1) for x in b)
    nt = (n + b.shape[1] - 1) // b.shape[1]
    h = (torch.linspace(-4.0, 4.0, nt, **f64) * (math.pi / 12)).view(-1, 1)
    sh, ch = torch.sin(h), torch.cos(h)
    u = (bx * sh + by * ch).reshape(-1)[:n]
    v = (-math.sin(dec) * (bx * ch - by * sh) + math.cos(dec) * bz).reshape(-1)[:n]
    w = (math.cos(dec) * (bx * ch - by * sh) + math.sin(dec) * bz).reshape(-1)[:n]
    return u.contiguous(), v.contiguous(), w.contiguous(), float(w.abs().max()) + 1e-9


def _samples(case, seed):
    """Samples normalised as the reference's inputs, on the device; span = 2*max(nx, ny)
    wavelengths, the longest baseline at 0.45 of the grid's extent along each axis."""
    n, nx, ny, F, P = (case[k] for k in ("n", "nx", "ny", "F", "P"))
    g = _gen(seed, 1)
    f64 = dict(dtype=torch.float64, device=DEV)
    a, b, c, wtop = _tracks(n, seed) if case["coverage"] == "tracks" else _disk(n, g)
    span = 2.0 * max(nx, ny)
    wmax = wtop * 0.45 * span
    d = dict(resolution=1.0 / int(span), wmin=-wmax, wmax=wmax)
    d["uu"] = 0.45 * a + 0.5
    d["vv"] = (0.45 * b + 0.5) * (ny / nx)
    d["ww"] = torch.clamp(0.5 * c / wtop + 0.5, 0.0, 1.0 - 2.0 ** -52)
    ul, vl, wl = (0.45 * span * x for x in (a, b, c))
    q2 = ul * ul + vl * vl
    host = np.random.default_rng(seed)
    sky_re = torch.zeros(n, **f64)
    sky_im = torch.zeros(n, **f64)
    for _ in range(2):
        l, m = host.uniform(-0.2, 0.2, 2)
        amp = host.uniform(0.5, 2.0) * torch.exp(
            -2 * math.pi ** 2 * host.uniform(1e-3, 5e-3) ** 2 * q2)
        ph = -2 * math.pi * (ul * l + vl * m + wl * (math.sqrt(1 - l * l - m * m) - 1))
        sky_re += amp * torch.cos(ph)
        sky_im += amp * torch.sin(ph)
    f32 = dict(dtype=torch.float32, device=DEV)
    fp = F * P
    d["vis_real"] = (sky_re.float().view(-1, 1) +
                     0.1 * torch.randn((n, fp), generator=g, **f32)).reshape(-1)
    d["vis_img"] = (sky_im.float().view(-1, 1) +
                    0.1 * torch.randn((n, fp), generator=g, **f32)).reshape(-1)
    if case["flagged"] > 0:
        d["vis_real"][torch.rand(n * fp, generator=g, **f32) < case["flagged"]] = float("nan")
    d["weight"] = 0.5 + torch.rand(n * P, generator=g, **f32)
    return d


def _sky(case, seed):
    """A sky image: compact sources over faint noise (float64 real and imaginary parts)."""
    nx, ny = case["nx"], case["ny"]
    g = _gen(seed, 2)
    f64 = dict(dtype=torch.float64, device=DEV)
    re = 1e-3 * torch.randn((ny, nx), generator=g, **f64)
    im = 1e-3 * torch.randn((ny, nx), generator=g, **f64)
    host = np.random.default_rng(seed + 1)
    y = torch.arange(ny, **f64).view(-1, 1)
    x = torch.arange(nx, **f64).view(1, -1)
    for _ in range(4):
        cy, cx = host.uniform(0.1, 0.9) * ny, host.uniform(0.1, 0.9) * nx
        s = host.uniform(1.5, 5.0)
        re += host.uniform(0.3, 1.5) * (torch.exp(-(y - cy) ** 2 / (2 * s * s)) *
                                        torch.exp(-(x - cx) ** 2 / (2 * s * s)))
    return re, im


FIELDS = ("uu", "vv", "ww", "vis_real", "vis_img", "weight")


def prepare(case, seed):
    nx, ny, nw = case["nx"], case["ny"], case["nw"]
    s = dict(case=case, **_samples(case, seed))
    kind = case["kind"]
    if kind == "dropin":
        for k in FIELDS:
            s[k] = s[k].cpu().numpy()
        s["grid"] = np.zeros(2 * nw * ny * nx)
        s["gridss"] = np.zeros(2 * nw * ny * nx)
        s["re"], s["im"] = np.zeros(ny * nx), np.zeros(ny * nx)
        return s
    cube = torch.empty((nw, ny, nx), dtype=imager.cube_dtype(case["precision"]), device=DEV)
    if kind == "image":
        s["cube"] = cube
        s["re"] = torch.empty((ny, nx), dtype=torch.float64, device=DEV)
        s["im"] = torch.empty_like(s["re"])
        return s
    s["x_re"], s["x_im"] = _sky(case, seed)
    if kind == "degrid":
        s["cube"] = cube
        dt = torch.float64 if case["precision"] == "fp64" else torch.float32
        s["m_re"] = torch.empty(case["n"], dtype=dt, device=DEV)
        s["m_im"] = torch.empty_like(s["m_re"])
        return s
    s["op"] = autograd.ImagingOperator(s["uu"], s["vv"], s["ww"], None, nw, case["support"], nx,
                                       ny, s["resolution"], s["wmin"], s["wmax"],
                                       precision=case["precision"], cube=cube)
    s["op"].plan()  # the samples' sort, kept over the iterations of a fit
    s["x_re"].requires_grad_(True)
    s["x_im"].requires_grad_(True)
    return s


def run(state):
    s, c = state, state["case"]
    nx, ny, nw, support = c["nx"], c["ny"], c["nw"], c["support"]
    if c["kind"] == "image":
        imager.image(*(s[k] for k in FIELDS), nw, support, nx, ny, s["resolution"], s["wmin"],
                     s["wmax"], precision=c["precision"], cube=s["cube"], image_real=s["re"],
                     image_imag=s["im"], freq_per_chan=c["F"], polarizations=c["P"])
        return {"re": s["re"], "im": s["im"]}
    if c["kind"] == "degrid":
        imager.degrid(s["x_re"], s["x_im"], s["uu"], s["vv"], s["ww"], s["weight"], nw, support,
                      s["resolution"], s["wmin"], s["wmax"], precision=c["precision"],
                      cube=s["cube"], model_real=s["m_re"], model_imag=s["m_im"])
        return {"m_re": s["m_re"], "m_im": s["m_im"]}
    if c["kind"] == "fit":
        s["x_re"].grad = s["x_im"].grad = None
        m_re, m_im = autograd.measure(s["x_re"], s["x_im"], s["op"])
        loss = autograd.chi2(m_re, m_im, s["vis_real"], s["vis_img"], s["weight"])
        loss.backward()
        return {"m_re": m_re.detach(), "m_im": m_im.detach(), "chi2": loss.detach(),
                "g_re": s["x_re"].grad, "g_im": s["x_im"].grad}
    for k in ("grid", "re", "im"):
        s[k].fill(0.0)
    imager.wstack(nw, c["n"], c["F"], c["P"], *(s[k] for k in FIELDS), 1.0 / nx, 1.0 / nw,
                  support, nx, ny, s["grid"])
    imager.fftw_data(s["grid"], s["gridss"], nx, ny, nw)
    imager.phase_correction(s["gridss"], s["re"], s["im"], nx, ny, nw, nx, ny, s["resolution"],
                            s["wmin"], s["wmax"])
    return {"re": s["re"], "im": s["im"]}


def work(case):
    """One pass: the samples (and for the adjoint the image) read once, the outputs written
    once; window updates, plane transforms and phase products.  The cube is scratch."""
    n, nx, ny, nw, F, P = (case[k] for k in ("n", "nx", "ny", "nw", "F", "P"))
    out = 8 if case["precision"] == "fp64" else 4
    samples = 24 * n + 8 * n * F * P + 4 * n * P
    image = 16 * nx * ny
    cells = nw * nx * ny
    one = n * case["support"] ** 2 * 4 + cells * (5 * math.log2(nx * ny) + 8)
    if case["kind"] == "degrid":
        return {"bytes": 28 * n + image + 2 * out * n, "flops": one}
    if case["kind"] == "fit":
        return {"bytes": samples + 2 * image + 2 * out * n, "flops": 2 * one}
    return {"bytes": samples + image, "flops": one}


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch

class _Exact:
    CHUNK = 1 << 22

    def __init__(self, case, s):
        self.nx, self.ny, self.nw = case["nx"], case["ny"], case["nw"]
        self.K = (case["support"] - 1) // 2
        self.s = s
        nx, ny, nw = self.nx, self.ny, self.nw
        self.gw = (s["ww"] / (1.0 / nw)).to(torch.int16)
        f64 = dict(dtype=torch.float64, device=DEV)

        def coord(m):
            i = torch.arange(m, **f64) - m // 2
            i = torch.where(i < 0, i + 2 * (m // 2), i)
            return torch.sin(i * s["resolution"])

        x, y = coord(nx).view(1, -1), coord(ny).view(-1, 1)
        self.fac = torch.sqrt(1 - (x * x + y * y))

    def planes(self):
        for w in range(self.nw):
            yield w, torch.nonzero(self.gw == w).view(-1)

    def axis(self, pos, size):
        """First cell and last cell of the windows, and the positions' cells."""
        K, g = self.K, pos.to(torch.int64)
        lo = torch.where(g > K - 1, g - K, torch.zeros_like(g))
        hi = torch.where(g < size - K, g + K, torch.full_like(g, size - 1))
        return lo, hi

    def windows(self, idx):
        """(flat cell, weight) of every window offset of samples idx; weight 0 outside."""
        pu = self.s["uu"][idx] / (1.0 / self.nx)
        pv = self.s["vv"][idx] / (1.0 / self.nx)
        j0, j1 = self.axis(pu, self.nx)
        k0, k1 = self.axis(pv, self.ny)
        for b in range(2 * self.K + 1):
            k = k0 + b
            ev = torch.where(k <= k1, torch.exp(-0.5 * (k + 0.5 - pv) ** 2), 0.0)
            for a in range(2 * self.K + 1):
                j = j0 + a
                eu = torch.where(j <= j1, torch.exp(-0.5 * (j + 0.5 - pu) ** 2), 0.0)
                cell = torch.clamp(k, max=self.ny - 1) * self.nx + torch.clamp(j, max=self.nx - 1)
                yield cell, (0.5 / PI_REF) * ev * eu

    def screen(self, w):
        """dwnorm*sqrt(1-r^2) and the angle of plane w; None for a single plane."""
        if self.nw == 1:
            return None
        dw = (self.s["wmax"] - self.s["wmin"]) / self.nw
        f = self.fac * (dw / (self.s["wmax"] - self.s["wmin"]))
        return torch.polar(f, 2 * PI_REF * (self.s["wmin"] + w * dw) * (self.fac - 1.0))

    def image(self, vr, vi):
        """Dirty image of summed weighted visibilities (float64, one per sample)."""
        nx, ny = self.nx, self.ny
        out = torch.zeros((ny, nx), dtype=torch.complex128, device=DEV)
        for w, idx in self.planes():
            re = torch.zeros(ny * nx, dtype=torch.float64, device=DEV)
            im = torch.zeros_like(re)
            for part in idx.split(self.CHUNK):
                pr, pi = vr[part], vi[part]
                for cell, cw in self.windows(part):
                    re.index_add_(0, cell, cw * pr)
                    im.index_add_(0, cell, cw * pi)
            plane = torch.fft.ifft2(torch.complex(re, im).view(ny, nx))
            z = self.screen(w)
            out += plane if z is None else plane * z
        return out.real.contiguous(), out.imag.contiguous()

    def degrid(self, x_re, x_im, weight):
        n = weight.numel()
        mr = torch.zeros(n, dtype=torch.float64, device=DEV)
        mi = torch.zeros_like(mr)
        x = torch.complex(x_re, x_im)
        for w, idx in self.planes():
            z = self.screen(w)
            plane = torch.fft.fft2(x if z is None else x * z.conj()).view(-1)
            plane = plane / (self.nx * self.ny)
            re, im = plane.real.contiguous(), plane.imag.contiguous()
            for part in idx.split(self.CHUNK):
                ar = torch.zeros(part.numel(), dtype=torch.float64, device=DEV)
                ai = torch.zeros_like(ar)
                for cell, cw in self.windows(part):
                    ar += cw * re[cell]
                    ai += cw * im[cell]
                wt = weight[part].double()
                mr[part] = wt * ar
                mi[part] = wt * ai
        return mr, mi


def exact(case, seed):
    with torch.no_grad():
        s = _samples(case, seed)
        e = _Exact(case, s)
        n, F, P = case["n"], case["F"], case["P"]
        if case["kind"] in ("image", "dropin"):
            # the float product weight*vis of the reference (w-stacking_omp.c:118-133), summed
            # in 64 bits; a NaN real part takes its visibility out
            wt = s["weight"].view(n, 1, P)
            vr, vi = s["vis_real"].view(n, F, P), s["vis_img"].view(n, F, P)
            keep = ~torch.isnan(vr)
            sr = torch.where(keep, wt * vr, 0.0).double().sum((1, 2))
            si = torch.where(keep, wt * vi, 0.0).double().sum((1, 2))
            re, im = e.image(sr, si)
            if case["kind"] == "dropin":
                re, im = re.view(-1).cpu().numpy(), im.view(-1).cpu().numpy()
            return {"re": re, "im": im}
        x_re, x_im = _sky(case, seed)
        if case["kind"] == "degrid":
            m_re, m_im = e.degrid(x_re, x_im, s["weight"])
            return {"m_re": m_re, "m_im": m_im}
        m_re, m_im = e.degrid(x_re, x_im, torch.ones_like(s["weight"]))
        dr = s["vis_real"].double() - m_re
        di = s["vis_img"].double() - m_im
        w = s["weight"].double()
        g_re, g_im = e.image(-2 * w * dr, -2 * w * di)
        return {"m_re": m_re, "m_im": m_im, "chi2": (w * (dr * dr + di * di)).sum(),
                "g_re": g_re, "g_im": g_im}
