"""Imaging float64 visibilities through an FP64 plan: against the sum of the images of their
float32 parts, with channels, flagged samples, dense tiles and windows wider than the tiles
take; and what it refuses."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nx,ny,nw,support,F,P", [(1, 64, 64, 2, 7, 1, 1),
                                                    (5000, 300, 200, 3, 7, 2, 2),
                                                    (20000, 128, 256, 4, 9, 1, 1),
                                                    (3000, 128, 128, 2, 21, 1, 2)])
def test_matches_the_float_parts(cuda, n, nx, ny, nw, support, F, P):
    """Both sides sum products weight*vis rounded to 53 bits (weights are powers of two here,
    so the float products of the parts are exact): 1e-12 relative L2."""
    import torch
    from lofar_amd import imager
    rng = np.random.default_rng(n)
    t = [torch.from_numpy(a).to(cuda) for a in (
        rng.uniform(0.3, 0.6, n), rng.uniform(0.3, 0.6, n) * ny / nx, rng.uniform(0, 0.999, n))]
    wt = torch.from_numpy(2.0 ** rng.integers(-2, 3, n * P).astype(np.float32)).to(cuda)
    vr = torch.from_numpy(rng.standard_normal(n * F * P)).to(cuda)
    vi = torch.from_numpy(rng.standard_normal(n * F * P)).to(cuda)
    if n > 1:
        vr[::17] = float("nan")  # skipped, as in float
    plan = imager.Plan(*t, wt, nw, support, nx, ny, freq_per_chan=F, polarizations=P)
    args = (1.0 / (2 * max(nx, ny)), -50.0, 80.0)
    re, im = plan.image64(vr, vi, wt, *args)
    hr, hi = vr.float(), vi.float()
    a, b = plan.image(hr, hi, wt, *args)
    plan.image((vr - hr).float(), (vi - hi).float(), wt, *args, image_real=a, image_imag=b,
               accumulate=True)
    want, got = torch.complex(a, b), torch.complex(re, im)
    assert float((got - want).abs().pow(2).sum().sqrt()) <= 1e-12 * float(
        want.abs().pow(2).sum().sqrt())


def test_refuses_other_plans_and_types(cuda):
    import torch
    from lofar_amd import LofarError, imager
    n = 100
    u = torch.rand(n, dtype=torch.float64, device=cuda)
    wt = torch.ones(n, device=cuda)
    v64 = torch.zeros(n, dtype=torch.float64, device=cuda)
    args = (1.0 / 128, -5.0, 5.0)
    with pytest.raises(LofarError):
        imager.Plan(u, u, u * 0.9, wt, 2, 7, 64, 64, precision="fp32c").image64(v64, v64, wt, *args)
    plan = imager.Plan(u, u, u * 0.9, wt, 2, 7, 64, 64)
    with pytest.raises(TypeError):
        plan.image(v64, v64, wt, *args)
    with pytest.raises(TypeError):
        plan.image64(v64.float(), v64.float(), wt, *args)
    with pytest.raises(ValueError):
        plan.image64(v64[:50].contiguous(), v64, wt, *args)


@pytest.mark.parametrize("n,nx,ny,nw,support,F,P", [(60000, 128, 256, 4, 9, 1, 1),
                                                    (20000, 64, 64, 1, 7, 2, 2)])
def test_dense_tiles_match_the_float_parts(cuda, n, nx, ny, nw, support, F, P):
    """The same with more than 4096 entries in several tiles, or in the only one: tiles that
    several workgroups sum."""
    test_matches_the_float_parts(cuda, n, nx, ny, nw, support, F, P)
