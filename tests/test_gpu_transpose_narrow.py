"""GPU: transposes on grids narrower than the field of view (ny < nx).  The rays that
enter outside run along the border rows of Siddon's, whose views go in parts; grids of
few slices scatter.
"""
import numpy as np
import pytest
import torch

from oracle_ffi import Geometry, Oracle
from test_gpu_parity import dev, rel_l2, to_desc
from tomogpi_amd import lib

pytestmark = pytest.mark.gpu


def _geom(nx, ny, nz, nu, nv, nphi, pixel=2.0):
    return Geometry(fod=2.0 * nx, fdd=4.0 * nx, nphi=nphi, su=nu * pixel, sv=nv * pixel, nu=nu, nv=nv, sx=float(nx),
                    sy=float(ny), sz=float(nz), nx=nx, ny=ny, nz=nz, num_start=1.0, den_start=7.0, num_stop=15.0,
                    den_stop=8.0)


# A scattered Siddon chord is the difference of two FP32 path parameters: up to
# 2 nx 2^-24 of itself, 1e-5 on 96 voxels, taken over the 40 chords and more that
# a voxel of the smallest problem here sums; the gathers' and the other operators'
# terms are each within a few 2^-24.
@pytest.mark.parametrize("nx,ny,nz,nu,nv,nphi", [
    (40, 24, 12, 40, 12, 33),                            # as wide as one wave's rows take, views in one part
    (41, 24, 12, 40, 13, 33), (41, 24, 13, 40, 13, 5),   # one more; five views are one part, too
    (48, 8, 20, 48, 20, 67), (48, 8, 20, 48, 21, 65),    # parts of 8 views, the last of 3 or one; the middle row
    (50, 1, 30, 50, 30, 40), (50, 2, 30, 50, 31, 40),    # one border row, nothing between two
    (37, 9, 270, 37, 60, 20), (60, 3, 66, 60, 64, 130),  # two z blocks, two steps of 64
    (64, 16, 1, 64, 1, 64), (64, 16, 4, 64, 4, 64), (96, 12, 1, 96, 40, 40), (64, 2, 1, 64, 8, 64),  # few slices
])
@pytest.mark.parametrize("op", ["siddon", "rs", "vi"])
def test_narrow_transposes(ctx, op, nx, ny, nz, nu, nv, nphi):
    g = _geom(nx, ny, nz, nu, nv, nphi)
    print(f"[case] {op} {nx} {ny} {nz} / {nu} {nv} {nphi}", flush=True)
    G, o, rng = lib.Geometry(ctx, to_desc(g)), Oracle(g), np.random.default_rng(nx)
    try:
        if op == "vi":
            x = rng.random(g.vol_shape, dtype=np.float32)
            out, ref = torch.full(g.sino_shape, np.nan, dtype=torch.float32, device="cuda"), o.vi_T(x)
            G.backproject_adjoint(dev(x), out)
        else:
            y = rng.random(g.sino_shape, dtype=np.float32)
            out = torch.full(g.vol_shape, np.nan, dtype=torch.float32, device="cuda")
            ref = o.siddon_T(y) if op == "siddon" else o.rs_T(y)
            G.project_adjoint(dev(y), out, lib.PROJ_SIDDON if op == "siddon" else lib.PROJ_RS)
        assert rel_l2(out.cpu().numpy(), ref) < 2e-6, rel_l2(out.cpu().numpy(), ref)
    finally:
        G.close()


def test_siddon_parts_of_64(ctx):
    test_narrow_transposes(ctx, "siddon", 700, 20, 3, 700, 6, 70)
