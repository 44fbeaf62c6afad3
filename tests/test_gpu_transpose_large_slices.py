"""GPU: slices of 2^26 voxels and more (256 MiB each), whose voxel columns are more
work items than one grid dimension takes."""
import pytest
import torch

from oracle_ffi import Geometry
from test_gpu_parity import to_desc
from tomogpi_amd import lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("op", ["siddon", "rs"])
def test_large_slices(ctx, op):
    """Every voxel is written, and <A x, y> = <x, A^T y> within 1e-5, as for the
    transposes' view chunks."""
    n, nz, nu, nv, nphi = 8200, 3, 48, 6, 2
    g = Geometry(fod=0.75 * n, fdd=1.5 * n, nphi=nphi, su=nu * 300.0, sv=nv * 2.0, nu=nu, nv=nv, sx=float(n), sy=float(n),
                 sz=float(nz), nx=n, ny=n, nz=nz, num_start=0.25, den_start=1.0, num_stop=1.5, den_stop=1.0)
    print(f"[case] {op} {n} x {n} x {nz}", flush=True)
    G = lib.Geometry(ctx, to_desc(g))
    proj = lib.PROJ_SIDDON if op == "siddon" else lib.PROJ_RS
    try:
        gen = torch.Generator(device="cuda").manual_seed(6)
        x = torch.rand(g.vol_shape, generator=gen, device="cuda")
        y = torch.rand(g.sino_shape, generator=gen, device="cuda")
        ax, aty = torch.empty_like(y), torch.full_like(x, float("nan"))
        G.project(x, ax, proj)
        G.project_adjoint(y, aty, proj)
        assert not torch.isnan(aty).any()
        lhs, rhs = lib.dot(ctx, ax, y), lib.dot(ctx, x, aty)
        assert abs(lhs - rhs) <= 1e-5 * abs(rhs), (lhs, rhs)
    finally:
        G.close()
