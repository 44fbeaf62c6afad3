"""GPU: the projectors' wave shapes at their edges, bit for bit against the oracle.

A wave holds 64, 32 or 16 detector rows of one or a few columns, picked from
the detector's row count, and a Siddon workgroup four consecutive views; the
sizes below lie on both sides of each rule and of each remainder.
"""
import numpy as np
import pytest
import torch

from oracle_ffi import Geometry, Oracle, scaled_geometry
from test_gpu_parity import dev, rel_l2, to_desc
from tomogpi_amd import lib

pytestmark = pytest.mark.gpu


def _check(ctx, g, op, dt):
    print(f"[case] {op} {dt} nu={g.nu} nv={g.nv} nphi={g.nphi} nz={g.nz}", flush=True)
    G = lib.Geometry(ctx, to_desc(g))
    try:
        v = dev(np.random.default_rng(g.nv).random(g.vol_shape, dtype=np.float32))
        if dt != "f32":
            v = v.to(torch.bfloat16 if dt == "bf16" else torch.float16)
        vol = v.float().cpu().numpy()
        o = Oracle(g)
        ref = o.siddon(vol) if op == "siddon" else o.rs(vol, cube=op == "rs_cube")
        proj = lib.PROJ_SIDDON if op == "siddon" else lib.PROJ_RS
        for extra in (0, lib.FLAG_INDEX_READS):
            out = torch.full(g.sino_shape, np.nan, dtype=torch.float32, device="cuda")
            G.project(v, out, proj, extra | (lib.FLAG_RS_FOV_CUBE if op == "rs_cube" else 0))
            got = out.cpu().numpy()
            assert np.array_equal(got, ref), (extra, rel_l2(got, ref))
    finally:
        G.close()


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("nv,nu,nphi,nz", [
    (1, 5, 1, 1), (15, 9, 3, 17), (16, 33, 4, 16), (17, 8, 5, 63), (31, 7, 2, 64), (33, 65, 7, 65), (56, 16, 4, 30),
    (57, 17, 6, 31), (63, 3, 9, 62), (64, 64, 8, 66), (65, 12, 3, 20), (130, 10, 5, 129),
])
def test_siddon_wave_shapes(ctx, nv, nu, nphi, nz, dt):
    g = Geometry(fod=90.0, fdd=180.0, nphi=nphi, su=nu * 2.0, sv=nv * 1.6, nu=nu, nv=nv, sx=37.0, sy=33.0, sz=float(nz),
                 nx=37, ny=33, nz=nz, num_start=1.0, den_start=7.0, num_stop=15.0, den_stop=8.0)
    _check(ctx, g, "siddon", dt)


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("op", ["rs", "rs_cube"])
@pytest.mark.parametrize("nv,nu,nphi,nz,ny", [
    (1, 5, 1, 1, 33), (15, 9, 3, 62, 37), (28, 8, 5, 63, 12), (29, 17, 4, 64, 37), (33, 65, 7, 65, 40), (70, 10, 6, 126, 37),
])
def test_rs_wave_shapes(ctx, nv, nu, nphi, nz, ny, op, dt):
    """Waves of 16 and 32 rows; volumes narrower than the FOV in y (samples off
    the grid, tested one by one) and not (untested up to the shortest ray)."""
    g = Geometry(fod=90.0, fdd=180.0, nphi=nphi, su=nu * 2.0, sv=nv * 1.6, nu=nu, nv=nv, sx=37.0, sy=float(ny),
                 sz=float(nz), nx=37, ny=ny, nz=nz, num_start=1.0, den_start=7.0, num_stop=15.0, den_stop=8.0)
    _check(ctx, g, op, dt)


@pytest.mark.parametrize("nz", [40, 41])
def test_siddon_steep_rays(ctx, nz):
    """Rays up to 70 degrees off the mid plane: several z planes per in-plane
    cell (the general step), in the waves that hold them; and both z
    directions in one wave (41 rows)."""
    g = Geometry(fod=40.0, fdd=60.0, nphi=6, su=60.0, sv=330.0, nu=30, nv=41, sx=24.0, sy=24.0, sz=float(nz), nx=24,
                 ny=24, nz=nz, num_start=0.0, den_start=1.0, num_stop=2.0, den_stop=1.0)
    _check(ctx, g, "siddon", "f32")


def test_siddon_column_runs(ctx):
    """A detector wide enough that each of the eight column runs holds several groups, row bands and view groups."""
    _check(ctx, scaled_geometry(48, 37, nu=150, nv=70), "siddon", "f32")


@pytest.mark.parametrize("nx,ny", [(64, 31), (31, 64), (64, 63)])
def test_siddon_narrow_grid(ctx, nx, ny):
    """A grid narrower than the FOV in y: rays enter the FOV outside it, cross
    several z planes before their first x or y plane (the border voxel's
    stretch), and do so in their second cell where the first crossing is x's."""
    g = Geometry(fod=80.0, fdd=160.0, nphi=48, su=64 * 2.0, sv=64 * 2.4, nu=64, nv=64, sx=float(nx), sy=float(ny),
                 sz=70.0, nx=nx, ny=ny, nz=70, num_start=0.0, den_start=1.0, num_stop=2.0, den_stop=1.0)
    _check(ctx, g, "siddon", "f32")
