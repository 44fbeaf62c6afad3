"""GPU: the transposes on acquisitions other than 1 mm voxels and a detector at
twice the source's distance, against the FP64-accumulating oracle (rel-L2 <=
1e-6: FP32 sums of at most a few thousand terms of one sign, each within a few
1e-7 of the oracle's).
"""
import numpy as np
import pytest
import torch

from oracle_ffi import Geometry, Oracle
from test_gpu_parity import dev, rel_l2, to_desc
from tomogpi_amd import lib

pytestmark = pytest.mark.gpu


def _geom(nx, ny, nz, nu, nv, nphi, pixel=2.0, fod=2.0, fdd=2.0, voxel=1.0, start=1.0 / 7.0, stop=1.875):
    """pixel in voxels at the detector, fod in volume widths, fdd in fod."""
    return Geometry(fod=fod * nx * voxel, fdd=fdd * fod * nx * voxel, nphi=nphi, su=nu * pixel * voxel,
                    sv=nv * pixel * voxel, nu=nu, nv=nv, sx=nx * voxel, sy=ny * voxel, sz=nz * voxel, nx=nx, ny=ny, nz=nz,
                    num_start=start, den_start=1.0, num_stop=stop, den_stop=1.0)


def _check(ctx, g, op, cube=False, bound=1e-6):
    print(f"[case] {op} {g.nx} {g.ny} {g.nz} / {g.nu} {g.nv} {g.nphi} fdd/fod {g.fdd / g.fod:.3g} voxel {g.sx / g.nx:.3g}",
          flush=True)
    G, o = lib.Geometry(ctx, to_desc(g)), Oracle(g)
    try:
        rng = np.random.default_rng(g.nz)
        if op == "vi":
            x = rng.random(g.vol_shape, dtype=np.float32)
            ref, out = o.vi_T(x), torch.full(g.sino_shape, np.nan, dtype=torch.float32, device="cuda")
            G.backproject_adjoint(dev(x), out)
        else:
            y = rng.random(g.sino_shape, dtype=np.float32)
            ref = o.siddon_T(y) if op == "siddon" else o.rs_T(y, cube=cube)
            out = torch.full(g.vol_shape, np.nan, dtype=torch.float32, device="cuda")
            G.project_adjoint(dev(y), out, lib.PROJ_SIDDON if op == "siddon" else lib.PROJ_RS,
                              lib.FLAG_RS_FOV_CUBE if cube else 0)
        assert rel_l2(out.cpu().numpy(), ref) <= bound
    finally:
        G.close()


@pytest.mark.parametrize("voxel", [0.1, 0.4, 0.55, 0.8, 1.1])
@pytest.mark.parametrize("nx,ny,nz,nu,nv,nphi", [(30, 31, 64, 40, 41, 65), (16, 16, 130, 24, 35, 40), (31, 30, 63, 40, 41, 30)])
@pytest.mark.parametrize("op", ["siddon", "vi", "rs"])
def test_voxel_size(ctx, op, nx, ny, nz, nu, nv, nphi, voxel):
    """Voxel sizes whose products round.  An odd number of rows over an even number of
    slices: the middle row's rays run along the plane between two slices and
    belong to the upper one alone."""
    _check(ctx, _geom(nx, ny, nz, nu, nv, nphi, voxel=voxel), op)


@pytest.mark.parametrize("fdd", [1.05, 1.2, 1.5])
@pytest.mark.parametrize("nx,ny,nz,nu,nv,nphi", [(30, 30, 30, 46, 46, 24), (24, 40, 33, 60, 40, 30), (40, 20, 24, 60, 33, 24)])
@pytest.mark.parametrize("op", ["siddon", "vi", "rs", "rs_cube"])
def test_detector_inside(ctx, op, nx, ny, nz, nu, nv, nphi, fdd):
    """A detector plane inside the volume (a virtual detector near the isocentre):
    the rays go on behind it, as the projector's."""
    _check(ctx, _geom(nx, ny, nz, nu, nv, nphi, pixel=0.8 * fdd, fdd=fdd), op.split("_")[0], cube=op == "rs_cube")


@pytest.mark.parametrize("nx,ny,nz,nv", [(32, 32, 24, 40), (30, 28, 33, 41), (64, 64, 20, 33), (31, 32, 24, 40), (128, 128, 6, 9)])
@pytest.mark.parametrize("voxel", [1.0, 0.55])
def test_siddon_rays_along_planes(ctx, nx, ny, nz, nv, voxel):
    """An odd number of detector columns over an even number of voxels: in the views
    along the axes the middle column's rays run along a plane between voxels, up
    to the rounding of the view's cosine, and belong to the voxels that the
    projector gives them to."""
    _check(ctx, _geom(nx, ny, nz, 41 if nx < 64 else 2 * (nx // 2) + 1, nv, 24, voxel=voxel, start=0.0, stop=2.0), "siddon")


@pytest.mark.parametrize("nx,ny,nz,nu,nv,nphi", [(20, 20, 20, 24, 16, 130), (24, 20, 70, 30, 16, 130), (20, 20, 3, 30, 15, 130)])
@pytest.mark.parametrize("op", ["siddon", "vi", "rs", "rs_cube"])
def test_few_fine_rows(ctx, op, nx, ny, nz, nu, nv, nphi):
    """Fewer detector rows than pass one voxel, and rays enough for the gather."""
    g = _geom(nx, ny, nz, nu, nv, nphi)
    g.sv = nv * 0.2
    _check(ctx, g, op.split("_")[0], cube=op == "rs_cube")


@pytest.mark.parametrize("op,nx,ny,nz,nu,nv,nphi", [
    ("siddon", 64, 64, 1, 64, 4, 64), ("siddon", 64, 64, 40, 64, 1, 300), ("rs", 64, 64, 1, 64, 16, 64),
    ("rs", 64, 64, 100, 64, 2, 64), ("vi", 64, 64, 1, 64, 1, 700),     # scattered: few rows or slices
    ("vi", 40, 40, 1, 40, 300, 30), ("vi", 40, 40, 2, 40, 301, 30), ("vi", 40, 40, 9, 40, 200, 30),  # rows off the volume
])
def test_thin(ctx, op, nx, ny, nz, nu, nv, nphi):
    """Rel-L2 <= 1e-5: the scatter adds FP32 terms one by one."""
    g = _geom(nx, ny, nz, nu, nv, nphi)
    _check(ctx, g, op, bound=1e-5)
