"""Mixed-radix transforms (sides with prime factors up to 13): every stage radix, lengths
with one to five stages, lines that do not fill a workgroup, and the allocation-free call's
device-filled twiddles, against numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


# lengths by their stages: one (3..15), two, three (13*13*13), four and five stages, the
# longest lines of each strip width, and powers of two beside another side
LENGTHS = [3, 5, 6, 7, 9, 10, 11, 12, 13, 15, 14, 22, 26, 33, 35, 49, 77, 121, 143, 169, 180, 225,
           240, 512, 1331, 2025, 2048, 2197, 2401, 3125, 4096, 6561, 7203, 8190, 8192]


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("other", [3, 10])
def test_every_radix_as_rows_and_columns(cuda, n, other):
    """Relative L2 against numpy in 64 bits: rounding grows like sqrt(log n) eps, far below
    1e-14 (FP64) and 2e-6 (FP32) at these lengths."""
    import torch
    from lofar_amd import imager
    rng = np.random.default_rng(n * 31 + other)
    for shape in ((2, n, other), (2, other, n)):
        x = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
        x32 = x.astype(np.complex64)
        for sign in (1, -1):
            f = np.fft.ifft2 if sign > 0 else lambda a, axes: np.fft.fft2(a, axes=axes) / (
                n * other)
            got = imager.fft(torch.from_numpy(x).to(cuda), sign=sign).cpu().numpy()
            assert rel(got, f(x, axes=(1, 2))) < 1e-14
            t = torch.from_numpy(x32).to(cuda)
            imager.fft(t, sign=sign, out=t)  # in place
            assert rel(t.cpu().numpy(), f(x32.astype(np.complex128), axes=(1, 2))) < 2e-6


@pytest.mark.parametrize("nx,ny", [(300, 480), (1000, 256)])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32c", 1e-6)])
def test_allocation_free_call_matches(cuda, nx, ny, precision, tol):
    """lofar_image_dev_static fills its twiddles on the device (sincospi, a few ulp from the
    host's): the image agrees to rounding."""
    import torch
    from lofar_amd import imager
    rng = np.random.default_rng(nx)
    n, nw = 20000, 3
    t = [torch.from_numpy(a).to(cuda) for a in (
        rng.uniform(0.1, 0.9, n), rng.uniform(0.1, 0.9, n) * ny / nx, rng.uniform(0, 0.999, n),
        rng.standard_normal(n).astype(np.float32), rng.standard_normal(n).astype(np.float32),
        rng.uniform(0.5, 1.5, n).astype(np.float32))]
    args = (nw, 7, nx, ny, 1.0 / (2 * max(nx, ny)), -40.0, 60.0)
    a = imager.image(*t, *args, precision=precision)
    b = imager.image(*t, *args, precision=precision, static_workspace=True)
    for p, q in zip(a, b):
        assert rel(q.cpu().numpy(), p.cpu().numpy()) < tol
