"""Sample counts at the edges of the bucket sort's chunk and block rules: one sample, a
workgroup's chunk and one more, and the counts where the chunk grows, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 511, 512, 513, 2049, 262144, 262145])
@pytest.mark.parametrize("nx,ny,nw", [(64, 64, 1), (200, 130, 3), (1100, 70, 2)])
def test_grid_and_degrid(cuda, n, nx, ny, nw):
    """FP64 cube within 1e-12 and FP32C within 1e-6 of the oracle's (relative L2), the
    interpolation at the same samples within 1e-12."""
    import torch
    from lofar_amd import imager
    rng = np.random.default_rng(n + nx)
    u = rng.uniform(-0.9 / nx, 1 + 2.0 / nx, n)
    v = rng.uniform(-0.9 / nx, (ny + 2.0) / nx, n)
    w = rng.uniform(0.0, 1 - 1e-12, n)
    vr = rng.standard_normal(n).astype(np.float32)
    vi = rng.standard_normal(n).astype(np.float32)
    wt = rng.uniform(0.2, 2.0, n).astype(np.float32)
    st, want = O.wstack(nw, u, v, w, vr, vi, wt, 1 / nx, 1 / nw, 7, nx, ny)
    assert st == O.OK
    t = [torch.from_numpy(a).to(cuda) for a in (u, v, w, vr, vi, wt)]
    for precision, tol in (("fp64", 1e-12), ("fp32c", 1e-6)):
        got = imager.grid(*t, nw, 7, nx, ny, precision=precision).cpu().numpy()
        assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want)
    cube = rng.standard_normal((nw, ny, nx)) + 1j * rng.standard_normal((nw, ny, nx))
    mr, mi = imager.degrid_cube(torch.from_numpy(cube).to(cuda), *t[:3], t[5], 7)
    st, ref = O.degrid(cube, u, v, w, wt, 1 / nx, 1 / nw, 7)
    assert st == O.OK
    got = mr.cpu().numpy() + 1j * mi.cpu().numpy()
    assert np.linalg.norm(got - ref) <= 1e-12 * np.linalg.norm(ref)
