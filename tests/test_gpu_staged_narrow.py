"""GPU: the LDS-staged projectors on grids narrower than the field of view, whose
rays enter it outside the grid: bit for bit against the oracle."""
import numpy as np
import pytest
import torch

from oracle_ffi import Geometry, Oracle
from test_gpu_parity import dev, rel_l2, to_desc
from tomogpi_amd import lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,nu,nv,nphi,pixel,fod,fdd", [
    (61, 34, 61, 122, 61, 40, 1.3, 0.6, 1.3), (67, 28, 67, 67, 69, 46, 0.7, 2.0, 1.3), (72, 41, 6, 72, 8, 56, 4.0, 2.0, 1.3),
    (90, 51, 60, 180, 40, 19, 2.0, 0.6, 1.3), (64, 12, 40, 64, 40, 30, 2.0, 2.0, 2.0), (40, 61, 40, 60, 50, 24, 2.0, 1.5, 2.0),
])
@pytest.mark.parametrize("op", ["siddon", "rs", "rs_cube"])
def test_staged_narrow_grid(ctx, op, nx, ny, nz, nu, nv, nphi, pixel, fod, fdd):
    g = Geometry(fod=fod * nx, fdd=fdd * fod * nx, nphi=nphi, su=nu * pixel, sv=nv * pixel, nu=nu, nv=nv, sx=float(nx),
                 sy=float(ny), sz=float(nz), nx=nx, ny=ny, nz=nz, num_start=0.3, den_start=1.0, num_stop=2.0, den_stop=1.0)
    print(f"[case] {op} {nx} {ny} {nz}", flush=True)
    G, o = lib.Geometry(ctx, to_desc(g)), Oracle(g)
    try:
        vol = np.random.default_rng(ny).random(g.vol_shape, dtype=np.float32)
        ref = o.siddon(vol) if op == "siddon" else o.rs(vol, cube=op == "rs_cube")
        out = torch.full(g.sino_shape, np.nan, dtype=torch.float32, device="cuda")
        G.project(dev(vol), out, lib.PROJ_SIDDON if op == "siddon" else lib.PROJ_RS,
                  lib.FLAG_STAGED | (lib.FLAG_RS_FOV_CUBE if op == "rs_cube" else 0))
        got = out.cpu().numpy()
        assert np.array_equal(got, ref), rel_l2(got, ref)
    finally:
        G.close()
