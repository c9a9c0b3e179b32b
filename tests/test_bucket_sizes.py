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


@pytest.mark.parametrize("n", [1, 511, 513, 1025, 262144, 262145, 524289])
def test_grid_and_degrid_two_levels(cuda, n):
    """576 tiles, more than one level sorts: the level-2 blocks' rule as well (1024 records up
    to 524288 samples, more beyond), with the tolerances above."""
    test_grid_and_degrid(cuda, n, 1500, 1500, 1)


CHILD = r"""
import hashlib, sys
import numpy as np, torch
from lofar_amd import imager
rng = np.random.default_rng(5)
n, nx, ny, nw = 30000, 200, 330, 4
t = [torch.from_numpy(a).cuda() for a in (
    rng.uniform(-0.01, 1.01, n), rng.uniform(-0.01, 1.01 * ny / nx, n), rng.uniform(0, 0.999, n),
    rng.standard_normal(n).astype(np.float32), rng.standard_normal(n).astype(np.float32),
    rng.uniform(0.5, 1.5, n).astype(np.float32))]
for p in ("fp64", "fp32c"):
    for support in (7, 17):
        c = imager.grid(*t, nw, support, nx, ny, precision=p)
        print(p, support, hashlib.sha256(c.cpu().numpy().tobytes()).hexdigest())
"""


def test_one_level_sort_gives_the_two_level_bits(cuda):
    """Few tiles are sorted by level 1 alone; LOFAR_BUCKET_CFG keeps both levels."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    outs = []
    for cfg in (None, "16,16384,8192", "2,1000,300"):
        env = dict(os.environ, PYTHONPATH=root)
        if cfg:
            env["LOFAR_BUCKET_CFG"] = cfg
        r = subprocess.run([sys.executable, "-c", CHILD], env=env, capture_output=True, text=True,
                           timeout=120)
        assert r.returncode == 0, r.stderr[-2000:]
        outs.append(r.stdout)
    # FP32C positions are rounded to the super-tile side's bits: the default's and the first
    # configuration's agree, the second's differ in FP32C only
    assert outs[0] == outs[1]
    assert outs[0].splitlines()[:2] == outs[2].splitlines()[:2]
