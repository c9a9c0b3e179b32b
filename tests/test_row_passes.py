"""The fused row passes where an image row's planes are split between groups of threads (short
rows of small images, four planes or more), on both sides of that rule and with plane counts
that do not divide, with the image accumulated, and their adjoint: against the oracle.
FP64 images within 1e-10 and FP32C within 1e-6 (relative L2), as at the other sizes."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nw", [(2, 4, 6), (16, 32, 9), (64, 64, 3), (64, 64, 4),
                                      (256, 256, 5), (512, 128, 7), (512, 1024, 4),
                                      (256, 2048, 4), (512, 256, 33), (1024, 64, 5)])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("fp32c", 1e-6)])
def test_image_and_adjoint(cuda, nx, ny, nw, precision, tol):
    import torch
    from lofar_amd import imager
    rng = np.random.default_rng(nx + nw)
    n = 4000
    u, v = rng.uniform(0.05, 0.95, n), rng.uniform(0.05, 0.95, n) * ny / nx
    w = rng.uniform(0.0, 1 - 1e-12, n)
    vr = rng.standard_normal(n).astype(np.float32)
    vi = rng.standard_normal(n).astype(np.float32)
    wt = rng.uniform(0.5, 1.5, n).astype(np.float32)
    res, wmin, wmax = 1.0 / (2 * max(nx, ny)), -60.0, 90.0
    want = O.image(nw, u, v, w, vr, vi, wt, 7, nx, ny, res, wmin, wmax)
    t = [torch.from_numpy(a).to(cuda) for a in (u, v, w, vr, vi, wt)]
    re, im = imager.image(*t, nw, 7, nx, ny, res, wmin, wmax, precision=precision)
    got = re.cpu().numpy() + 1j * im.cpu().numpy()
    assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want)
    imager.image(*t, nw, 7, nx, ny, res, wmin, wmax, precision=precision, image_real=re,
                 image_imag=im, accumulate=True)
    got = re.cpu().numpy() + 1j * im.cpu().numpy()
    assert np.linalg.norm(got - 2 * want) <= tol * np.linalg.norm(2 * want)
    y = rng.standard_normal((ny, nx)) + 1j * rng.standard_normal((ny, nx))
    ref = O.degrid_image(y, nw, u, v, w, wt, 7, res, wmin, wmax)
    mr, mi = imager.degrid(torch.from_numpy(y.real.copy()).to(cuda),
                           torch.from_numpy(y.imag.copy()).to(cuda), *t[:3], t[5], nw, 7, res,
                           wmin, wmax, precision=precision)
    got = mr.cpu().numpy() + 1j * mi.cpu().numpy()
    assert np.linalg.norm(got - ref) <= (1e-10 if precision == "fp64" else 1e-5) * \
        np.linalg.norm(ref)
