"""Plan.image64's length checks on the host: arrays shorter than the plan's samples need are
refused before anything reaches the library (CPU tensors, no device)."""
import pytest


@pytest.mark.parametrize("short", ["vis_real", "vis_img", "weight"])
@pytest.mark.parametrize("F,P", [(1, 1), (3, 2)])
def test_short_arrays_are_refused(short, F, P):
    import torch
    from lofar_amd import imager
    p = imager.Plan.__new__(imager.Plan)  # the fields alone: no sort on a device
    p.precision, p.n, p.F, p.P = imager.FP64, 50, F, P
    p.nw, p.nx, p.ny, p.device = 2, 64, 64, torch.device("cpu")
    need = {"vis_real": 50 * F * P, "vis_img": 50 * F * P, "weight": 50 * P}
    a = {k: torch.zeros(n - (k == short),
                        dtype=torch.float32 if k == "weight" else torch.float64)
         for k, n in need.items()}
    with pytest.raises(ValueError):
        p.image64(a["vis_real"], a["vis_img"], a["weight"], 1.0 / 128, -5.0, 5.0)
