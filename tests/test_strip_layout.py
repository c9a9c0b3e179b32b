"""Images go through strip-major scratch cubes; the separate passes keep row-major ones.  The
image against grid, fft and phase of the same samples, at one strip, less than one (row-major),
strips shorter and longer than a row pass's loads, rows of 8192 (two passes), few rows, row
counts that no XCD share divides, and mixed-radix sides with and without strips.  Both sides are the same sums: FP64 agrees to rounding
(1e-12), FP32C to two FP32 transforms' (2e-6); a misplaced cell is an error of order one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nw", [(8, 64, 3), (16, 16, 2), (32, 8, 5), (64, 512, 4),
                                      (128, 2, 3), (512, 64, 3), (1024, 4, 6), (2048, 128, 2),
                                      (4096, 64, 3), (16, 8192, 2), (8192, 2, 3),
                                      (8192, 64, 2), (12, 25, 3), (100, 7, 2), (300, 480, 3),
                                      (1250, 60, 2), (64, 90, 3), (1000, 2, 2), (3000, 66, 2)])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32c", 2e-6)])
def test_image_equals_the_separate_passes(cuda, nx, ny, nw, precision, tol):
    import torch
    from lofar_amd import imager
    rng = np.random.default_rng(nx + 3 * ny + nw)
    n = 3000
    t = [torch.from_numpy(a).to(cuda) for a in (
        rng.uniform(0.0, 0.999, n), rng.uniform(0.0, 0.999, n) * ny / nx,
        rng.uniform(0, 0.999, n), rng.standard_normal(n).astype(np.float32),
        rng.standard_normal(n).astype(np.float32), rng.uniform(0.5, 1.5, n).astype(np.float32))]
    geo = (1.0 / (2 * max(nx, ny)), -40.0, 60.0)
    cube = imager.grid(*t, nw, 7, nx, ny, precision=precision)
    want = torch.complex(*imager.phase(imager.fft(cube, sign=1), *geo))
    re, im = imager.image(*t, nw, 7, nx, ny, *geo, precision=precision)
    assert torch.linalg.norm(torch.complex(re, im) - want) <= tol * torch.linalg.norm(want)
    imager.image(*t, nw, 7, nx, ny, *geo, precision=precision, image_real=re, image_imag=im,
                 accumulate=True)
    assert torch.linalg.norm(torch.complex(re, im) - 2 * want) <= 2 * tol * torch.linalg.norm(want)
