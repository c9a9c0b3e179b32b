"""FP64 adjoints of unusual float64 cotangents: the planned call (one pass over doubles) against
the unplanned one (two passes over float parts) where products are NaN, and against itself at
other scales, in tiles summed by one workgroup and by several."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def samples(cuda, n, seed):
    import torch
    rng = np.random.default_rng(seed)
    return [torch.from_numpy(a).to(cuda) for a in (
        rng.uniform(0.2, 0.8, n), rng.uniform(0.2, 0.8, n), rng.uniform(0, 0.999, n),
        rng.standard_normal(n), rng.standard_normal(n))]


@pytest.mark.parametrize("support", [7, 21])
@pytest.mark.parametrize("n", [300, 20000])
def test_nan_products_are_skipped(cuda, n, support):
    """A visibility whose weighted real part is NaN (NaN weight, or 0 times infinity) adds
    nothing, with a plan and without: both sum 53-bit products, 1e-12 relative L2."""
    import torch
    from lofar_amd import autograd
    u, v, w, vr, vi = samples(cuda, n, n)
    wt = 0.5 + torch.rand(n, device=cuda)
    wt[::7] = float("nan")
    wt[1::7] = 0.0
    vr[1::14] = float("inf")
    out = []
    for plan in (False, True):
        op = autograd.ImagingOperator(u, v, w, wt, 2, support, 64, 64, 1.0 / 128, -40.0, 60.0,
                                      plan=plan)
        out.append(torch.complex(*op.adjoint(vr, vi)))
    assert torch.isfinite(torch.view_as_real(out[0])).all()
    assert torch.linalg.norm(out[1] - out[0]) <= 1e-12 * torch.linalg.norm(out[0])


@pytest.mark.parametrize("n", [300, 20000])
@pytest.mark.parametrize("scale", [-1000, -960, -900, -300, 900])
def test_image_scales_with_the_visibilities(cuda, n, scale):
    """Powers of two change no rounding above the smallest normal numbers, so the image of
    2^scale times the visibilities is 2^scale times theirs, to the two sums' rounding (1e-12
    relative L2; 2^-1000: the image's values, 2^-12 of the cells', keep 2^-1074 of 2^-1012,
    1e-12 as well)."""
    import torch
    from lofar_amd import imager
    u, v, w, vr, vi = samples(cuda, n, n + 1)
    one = torch.ones(n, device=cuda)
    plan = imager.Plan(u, v, w, one, 2, 7, 64, 64)
    args = (1.0 / 128, -40.0, 60.0)
    want = torch.complex(*plan.image64(vr, vi, one, *args))
    f = 2.0 ** scale
    re, im = plan.image64(vr * f, vi * f, one, *args)
    got = torch.complex(re * 2.0 ** -scale, im * 2.0 ** -scale)
    assert torch.linalg.norm(got - want) <= 1e-12 * torch.linalg.norm(want)
