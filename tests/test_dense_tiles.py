"""Dense tiles, split over several workgroups: gridding and degridding against the oracle at
the split's edges and for every kind of sum, bitwise independence of the sample order, and
plans bit for bit.

Tolerances (relative L2): the FP64 quantum is 2^-(60 - log2 of the entries touching the
densest 4x4 block) of the largest contribution, below 2^-44 here, and its rounding averages
over a cell's entries: 1e-12.  FP32C contributions are float products: 1e-6."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def case(n, nx, ny, nw, kind, seed=0):
    """n samples around the middle of tile (1, 0): over the tile, or in one cell's window."""
    rng = np.random.default_rng(seed + n)
    spread = 1.5 if kind == "point" else 24.0
    u = (96.0 + rng.uniform(-spread, spread, n)) / nx
    v = (32.0 + rng.uniform(-spread, spread, n)) / nx
    w = np.full(n, 0.5 / nw)
    vr = rng.standard_normal(n).astype(np.float32)
    vi = rng.standard_normal(n).astype(np.float32)
    if kind == "outlier":
        vr[n // 3] = 1e8
    if kind == "inf":
        vi[n // 2] = np.inf
    if kind == "zero":
        vr[:] = 0.0
        vi[:] = 0.0
    wt = rng.uniform(0.5, 1.5, n).astype(np.float32)
    return u, v, w, vr, vi, wt


def close(got, want, tol):
    ok = np.isfinite(want)
    assert np.array_equal(ok, np.isfinite(got))
    assert np.linalg.norm(got[ok] - want[ok]) <= tol * np.linalg.norm(want[ok])


@pytest.mark.parametrize("n", [4096, 4097, 8192, 8193, 12289, 70000])
@pytest.mark.parametrize("kind", ["spread", "point", "outlier", "inf", "zero"])
def test_grid_degrid_and_plan(cuda, n, kind):
    import torch
    from lofar_amd import imager
    nx, ny, nw = 130, 70, 2
    d = case(n, nx, ny, nw, kind)
    st, want = O.wstack(nw, *d, 1 / nx, 1 / nw, 7, nx, ny)
    assert st == O.OK
    t = [torch.from_numpy(a).to(cuda) for a in d]
    perm = torch.from_numpy(np.random.default_rng(1).permutation(n)).to(cuda)
    for precision, tol in (("fp64", 1e-12), ("fp32c", 1e-6)):
        got = imager.grid(*t, nw, 7, nx, ny, precision=precision)
        close(got.cpu().numpy(), want, tol)
        if kind in ("spread", "point", "zero"):  # integer sums: any order, the same bits
            again = imager.grid(*[x[perm].contiguous() for x in t], nw, 7, nx, ny,
                                precision=precision)
            assert torch.equal(torch.view_as_real(got), torch.view_as_real(again))
    cube = np.random.default_rng(2).standard_normal((nw, ny, nx)) + 0j
    st, ref = O.degrid(cube, *d[:3], d[5], 1 / nx, 1 / nw, 7)
    assert st == O.OK
    mr, mi = imager.degrid_cube(torch.from_numpy(cube).to(cuda), *t[:3], t[5], 7)
    close(mr.cpu().numpy() + 1j * mi.cpu().numpy(), ref, 1e-12)


@pytest.mark.parametrize("n", [20000, 80000])
@pytest.mark.parametrize("support", [5, 9, 13])
@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
def test_image_and_plan(cuda, n, support, precision):
    """The strip-major (FP64) and row-major cube of the fused path, and a plan, which keeps
    the list of dense tiles: twice with other visibilities, the bits of the unplanned call."""
    import torch
    from lofar_amd import imager
    nx, ny, nw = 256, 128, 2
    d = case(n, nx, ny, nw, "spread", seed=support)
    t = [torch.from_numpy(a).to(cuda) for a in d]
    args = (1.0 / 512, -40.0, 60.0)
    plan = imager.Plan(*t[:3], t[5], nw, support, nx, ny, precision=precision)
    tol = 1e-10 if precision == "fp64" else 1e-6
    for k in range(2):
        vr = (t[3] * (1.0 + k)).contiguous()
        re, im = imager.image(*t[:3], vr, t[4], t[5], nw, support, nx, ny, *args,
                              precision=precision)
        pre, pim = plan.image(vr, t[4], t[5], *args)
        assert torch.equal(re, pre) and torch.equal(im, pim)
        want = O.image(nw, *d[:3], vr.cpu().numpy(), *d[4:], support, nx, ny, *args)
        close(re.cpu().numpy() + 1j * im.cpu().numpy(), want, tol)
    sky = torch.randn((ny, nx), dtype=torch.float64, device=cuda)
    a = imager.degrid(sky, sky, *t[:3], t[5], nw, support, *args, precision=precision)
    b = plan.degrid(sky, sky, *args)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


@pytest.mark.parametrize("kind", ["spread", "point", "outlier", "inf"])
@pytest.mark.parametrize("nx,ny,nw", [(1100, 1000, 2), (1024, 1024, 3)])
def test_two_level_sort(cuda, nx, ny, nw, kind):
    """More than 512 tiles, so two levels sort them: the dense tile among sparse ones, its
    super-tile's records in more level-2 blocks than one read of the scan takes (70000 in
    blocks of 1024).  Grid, degridding, image and plan as above, with the same tolerances."""
    import torch
    from lofar_amd import imager
    n, sparse = 70000, 5000
    rng = np.random.default_rng(nx)
    back = (rng.uniform(0, 0.999, sparse), rng.uniform(0, 0.999, sparse) * ny / nx,
            rng.uniform(0, 0.999, sparse), rng.standard_normal(sparse).astype(np.float32),
            rng.standard_normal(sparse).astype(np.float32),
            rng.uniform(0.5, 1.5, sparse).astype(np.float32))
    d = [np.concatenate(x) for x in zip(case(n, nx, ny, nw, kind), back)]
    st, want = O.wstack(nw, *d, 1 / nx, 1 / nw, 7, nx, ny)
    assert st == O.OK
    cube = rng.standard_normal((nw, ny, nx)) + 0j
    st, ref = O.degrid(cube, *d[:3], d[5], 1 / nx, 1 / nw, 7)
    assert st == O.OK
    t = [torch.from_numpy(a).to(cuda) for a in d]
    perm = torch.from_numpy(np.random.default_rng(1).permutation(len(d[0]))).to(cuda)
    mr, mi = imager.degrid_cube(torch.from_numpy(cube).to(cuda), *t[:3], t[5], 7)
    close(mr.cpu().numpy() + 1j * mi.cpu().numpy(), ref, 1e-12)
    args = (1.0 / 2200, -40.0, 60.0)
    sky = torch.randn((ny, nx), dtype=torch.float64, device=cuda)
    for precision, tol in (("fp64", 1e-12), ("fp32c", 1e-6)):
        got = imager.grid(*t, nw, 7, nx, ny, precision=precision)
        close(got.cpu().numpy(), want, tol)
        plan = imager.Plan(*t[:3], t[5], nw, 7, nx, ny, precision=precision)
        a = imager.degrid(sky, sky, *t[:3], t[5], nw, 7, *args, precision=precision)
        b = plan.degrid(sky, sky, *args)
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
        if kind in ("outlier", "inf"):
            continue  # floating sums: no fixed order, and no finite image of an infinity
        again = imager.grid(*[x[perm].contiguous() for x in t], nw, 7, nx, ny,
                            precision=precision)
        assert torch.equal(torch.view_as_real(got), torch.view_as_real(again))
        re, im = imager.image(*t, nw, 7, nx, ny, *args, precision=precision)
        pre, pim = plan.image(*t[3:], *args)
        assert torch.equal(re, pre) and torch.equal(im, pim)
        img = O.image(nw, *d, 7, nx, ny, *args)
        close(re.cpu().numpy() + 1j * im.cpu().numpy(), img,
              1e-10 if precision == "fp64" else 1e-6)
