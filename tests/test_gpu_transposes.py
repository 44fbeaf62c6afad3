"""GPU: the gather forms of the transposes at the edges of their rules, against
the FP64-accumulating oracle (rel-L2 <= 1e-6: FP32 sums of at most a few
thousand terms of one sign, each within a few 1e-7 of the oracle's).
"""
import numpy as np
import pytest
import torch

from oracle_ffi import Geometry, Oracle
from test_gpu_parity import dev, rel_l2, to_desc
from tomogpi_amd import lib

pytestmark = pytest.mark.gpu


def _geom(nx, ny, nz, nu, nv, nphi, pixel=2.0, fod=2.0):
    return Geometry(fod=fod * nx, fdd=2.0 * fod * nx, nphi=nphi, su=nu * pixel, sv=nv * pixel, nu=nu, nv=nv, sx=float(nx),
                    sy=float(ny), sz=float(nz), nx=nx, ny=ny, nz=nz, num_start=1.0, den_start=7.0, num_stop=15.0,
                    den_stop=8.0)


def _geometry(ctx, g):
    print(f"[case] {g.nx} {g.ny} {g.nz} / {g.nu} {g.nv} {g.nphi}", flush=True)
    return lib.Geometry(ctx, to_desc(g))


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("nx,ny,nz,nu,nv,nphi,pixel", [
    (30, 30, 63, 40, 40, 20, 2.0), (30, 31, 64, 40, 41, 65, 2.0),   # one step of z; the middle row between two slices
    (31, 30, 65, 40, 40, 64, 2.0), (17, 33, 129, 33, 90, 31, 2.0),  # two, three steps; a grid narrower than the FOV
    (16, 16, 257, 24, 140, 20, 2.0), (64, 20, 24, 64, 33, 40, 2.0),  # two z blocks; much narrower
    (20, 20, 20, 90, 90, 12, 0.45), (24, 24, 24, 24, 24, 16, 2.0),  # many rows and columns a voxel; the scatter form
    (33, 1, 1, 50, 7, 70, 1.0), (1, 1, 40, 9, 60, 30, 1.0),         # one slice, one column
])
def test_siddon_transpose(ctx, nx, ny, nz, nu, nv, nphi, pixel, dt):
    g = _geom(nx, ny, nz, nu, nv, nphi, pixel)
    G = _geometry(ctx, g)
    try:
        y = dev(np.random.default_rng(nz).random(g.sino_shape, dtype=np.float32))
        if dt != "f32":
            y = y.to(torch.bfloat16 if dt == "bf16" else torch.float16)
        ref = Oracle(g).siddon_T(y.float().cpu().numpy())
        out = torch.full(g.vol_shape, np.nan, dtype=torch.float32, device="cuda")
        G.project_adjoint(y, out, lib.PROJ_SIDDON)
        assert rel_l2(out.cpu().numpy(), ref) <= 1e-6
    finally:
        G.close()


def test_siddon_transpose_source_inside(ctx):
    """A source inside the volume's bounding square (the scatter form)."""
    g = _geom(40, 40, 30, 40, 40, 24, pixel=1.0, fod=0.6)
    G = _geometry(ctx, g)
    try:
        y = np.random.default_rng(3).random(g.sino_shape, dtype=np.float32)
        out = torch.empty(g.vol_shape, dtype=torch.float32, device="cuda")
        G.project_adjoint(dev(y), out, lib.PROJ_SIDDON)
        assert rel_l2(out.cpu().numpy(), Oracle(g).siddon_T(y)) <= 1e-5
    finally:
        G.close()


def test_siddon_transpose_view_chunks(ctx):
    """More than 1 GiB of sinogram copy: the views go in two chunks that add
    (<A x, y> = <x, A^T y> within 1e-5)."""
    g = _geom(24, 24, 24, 1024, 1024, 260, pixel=0.08)
    G = _geometry(ctx, g)
    try:
        gen = torch.Generator(device="cuda").manual_seed(5)
        x = torch.rand(g.vol_shape, generator=gen, device="cuda")
        y = torch.rand(g.sino_shape, generator=gen, device="cuda")
        ax, aty = torch.empty_like(y), torch.empty_like(x)
        G.project(x, ax, lib.PROJ_SIDDON)
        G.project_adjoint(y, aty, lib.PROJ_SIDDON)
        lhs, rhs = lib.dot(ctx, ax, y), lib.dot(ctx, x, aty)
        assert abs(lhs - rhs) <= 1e-5 * abs(rhs), (lhs, rhs)
    finally:
        G.close()


def test_siddon_transpose_infinity(ctx):
    """An infinite sinogram cell reaches the voxels its ray crosses and no other."""
    g = _geom(32, 32, 40, 48, 48, 20)
    G = _geometry(ctx, g)
    try:
        y = np.random.default_rng(8).random(g.sino_shape, dtype=np.float32)
        one = np.zeros_like(y)
        one[7, 30, 20] = 1.0
        hit = Oracle(g).siddon_T(one) > 0.0
        y[7, 30, 20] = np.inf
        out = torch.empty(g.vol_shape, dtype=torch.float32, device="cuda")
        G.project_adjoint(dev(y), out, lib.PROJ_SIDDON)
        got = out.cpu().numpy()
        assert np.isfinite(got[~hit]).all()
        assert np.isinf(got[hit]).mean() > 0.99  # a chord of rounding length may count as none
    finally:
        G.close()


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("nx,ny,nz,nu,nv,nphi,pixel", [
    (30, 30, 30, 40, 63, 20, 2.0), (30, 31, 33, 41, 64, 21, 2.0), (31, 30, 40, 42, 65, 20, 2.0),  # one, two steps of rows
    (33, 17, 129, 17, 190, 31, 2.0), (16, 16, 200, 24, 256, 20, 2.0),  # three, four; partial column groups
    (16, 16, 180, 19, 257, 20, 2.0), (64, 20, 24, 64, 33, 40, 2.0),    # two row blocks; a narrow grid
    (20, 20, 20, 90, 90, 12, 0.3), (40, 40, 60, 9, 11, 30, 9.0),       # many cells a voxel, many voxels a cell
    (40, 40, 61, 30, 34, 30, 4.0), (33, 1, 1, 50, 7, 70, 1.0), (1, 1, 40, 9, 60, 30, 1.0),  # one slice, one column
    (20, 20, 20, 1, 1, 8, 3.0),
])
def test_vi_transpose(ctx, nx, ny, nz, nu, nv, nphi, pixel, dt):
    g = _geom(nx, ny, nz, nu, nv, nphi, pixel)
    G = _geometry(ctx, g)
    try:
        x = dev(np.random.default_rng(nz).random(g.vol_shape, dtype=np.float32))
        if dt != "f32":
            x = x.to(torch.bfloat16 if dt == "bf16" else torch.float16)
        ref = Oracle(g).vi_T(x.float().cpu().numpy())
        out = torch.full(g.sino_shape, np.nan, dtype=torch.float32, device="cuda")
        G.backproject_adjoint(x, out)
        assert rel_l2(out.cpu().numpy(), ref) <= 1e-6
    finally:
        G.close()


def test_vi_transpose_source_inside(ctx):
    """A source inside the volume's bounding square (the scatter form)."""
    g = _geom(40, 40, 30, 40, 40, 24, pixel=1.0, fod=0.6)
    G = _geometry(ctx, g)
    try:
        x = np.random.default_rng(3).random(g.vol_shape, dtype=np.float32)
        out = torch.empty(g.sino_shape, dtype=torch.float32, device="cuda")
        G.backproject_adjoint(dev(x), out)
        assert rel_l2(out.cpu().numpy(), Oracle(g).vi_T(x)) <= 1e-5
    finally:
        G.close()


def test_vi_transpose_infinity(ctx):
    """An infinite voxel reaches the cells around its projections and no other."""
    g = _geom(32, 32, 40, 48, 70, 20)
    G = _geometry(ctx, g)
    try:
        x = np.random.default_rng(8).random(g.vol_shape, dtype=np.float32)
        one = np.zeros_like(x)
        one[17, 30, 20] = 1.0
        hit = Oracle(g).vi_T(one) > 0.0
        x[17, 30, 20] = np.inf
        out = torch.empty(g.sino_shape, dtype=torch.float32, device="cuda")
        G.backproject_adjoint(dev(x), out)
        got = out.cpu().numpy()
        assert np.isfinite(got[~hit]).all()
        assert np.isinf(got[hit]).mean() > 0.99  # a weight of rounding size may count as none
    finally:
        G.close()


@pytest.mark.parametrize("op", ["siddon", "vi", "rs"])
def test_transpose_under_capture(ctx, op):
    """A captured transpose allocates nothing: the scatter form, replayed with new
    inputs against the eager call (1e-5: two FP32 sums of the same terms)."""
    g = _geom(48, 48, 48, 48, 48, 40)
    G = _geometry(ctx, g)
    try:
        a, b = (g.vol_shape, g.sino_shape) if op == "vi" else (g.sino_shape, g.vol_shape)
        x, y = torch.rand(a, device="cuda"), torch.empty(b, device="cuda")

        def run(out):
            if op == "vi":
                G.backproject_adjoint(x, out)
            else:
                G.project_adjoint(x, out, lib.PROJ_RS if op == "rs" else lib.PROJ_SIDDON)

        run(y)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            run(y)
        for _ in range(4):
            x.uniform_()
            y.fill_(np.nan)
            graph.replay()
            eager = torch.empty_like(y)
            run(eager)
            torch.cuda.synchronize()
            assert rel_l2(y.cpu().numpy(), eager.cpu().numpy()) <= 1e-5
    finally:
        G.close()


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("cube", [False, True])
@pytest.mark.parametrize("nx,ny,nz,nu,nv,nphi,pixel", [
    (30, 30, 63, 40, 40, 20, 2.0), (30, 31, 64, 40, 41, 65, 2.0),   # one step of z; views past 64
    (31, 30, 65, 40, 60, 64, 2.0), (17, 33, 129, 33, 90, 31, 2.0),  # two, three steps; a grid narrower than the FOV
    (16, 16, 257, 24, 140, 20, 2.0), (64, 20, 24, 64, 33, 40, 2.0),  # two z blocks; much narrower
    (20, 20, 20, 90, 90, 12, 0.45), (24, 24, 24, 12, 9, 16, 5.0),   # many rows and columns a voxel, few
    (33, 1, 1, 50, 7, 70, 1.0), (1, 1, 40, 9, 60, 30, 1.0),         # one slice, one column
])
def test_rs_transpose(ctx, nx, ny, nz, nu, nv, nphi, pixel, cube, dt):
    g = _geom(nx, ny, nz, nu, nv, nphi, pixel)
    G = _geometry(ctx, g)
    try:
        y = dev(np.random.default_rng(nz).random(g.sino_shape, dtype=np.float32))
        if dt != "f32":
            y = y.to(torch.bfloat16 if dt == "bf16" else torch.float16)
        ref = Oracle(g).rs_T(y.float().cpu().numpy(), cube=cube)
        out = torch.full(g.vol_shape, np.nan, dtype=torch.float32, device="cuda")
        G.project_adjoint(y, out, lib.PROJ_RS, lib.FLAG_RS_FOV_CUBE if cube else 0)
        got = out.cpu().numpy()
        if not ref.any():
            assert not got.any()
        else:
            assert rel_l2(got, ref) <= 1e-6
    finally:
        G.close()


def test_rs_transpose_source_inside(ctx):
    """A source inside the volume's bounding square (the scatter form)."""
    g = _geom(40, 40, 30, 40, 40, 24, pixel=1.0, fod=0.6)
    G = _geometry(ctx, g)
    try:
        y = np.random.default_rng(3).random(g.sino_shape, dtype=np.float32)
        out = torch.empty(g.vol_shape, dtype=torch.float32, device="cuda")
        G.project_adjoint(dev(y), out, lib.PROJ_RS)
        assert rel_l2(out.cpu().numpy(), Oracle(g).rs_T(y)) <= 1e-5
    finally:
        G.close()


def test_rs_transpose_view_chunks(ctx):
    """More than 1 GiB of the rays' table: the views go in two chunks that add
    (<A x, y> = <x, A^T y> within 1e-5)."""
    g = _geom(24, 24, 24, 1024, 1024, 80, pixel=0.08)
    G = _geometry(ctx, g)
    try:
        gen = torch.Generator(device="cuda").manual_seed(5)
        x = torch.rand(g.vol_shape, generator=gen, device="cuda")
        y = torch.rand(g.sino_shape, generator=gen, device="cuda")
        ax, aty = torch.empty_like(y), torch.empty_like(x)
        G.project(x, ax, lib.PROJ_RS)
        G.project_adjoint(y, aty, lib.PROJ_RS)
        lhs, rhs = lib.dot(ctx, ax, y), lib.dot(ctx, x, aty)
        assert abs(lhs - rhs) <= 1e-5 * abs(rhs), (lhs, rhs)
    finally:
        G.close()


def test_rs_transpose_infinity(ctx):
    """An infinite sinogram cell reaches the voxels around its samples and no other."""
    g = _geom(32, 32, 40, 48, 48, 20)
    G = _geometry(ctx, g)
    try:
        y = np.random.default_rng(8).random(g.sino_shape, dtype=np.float32)
        one = np.zeros_like(y)
        one[7, 30, 20] = 1.0
        hit = Oracle(g).rs_T(one) > 0.0
        y[7, 30, 20] = np.inf
        out = torch.empty(g.vol_shape, dtype=torch.float32, device="cuda")
        G.project_adjoint(dev(y), out, lib.PROJ_RS)
        got = out.cpu().numpy()
        assert np.isfinite(got[~hit]).all()
        assert np.isinf(got[hit]).mean() > 0.99  # a weight of rounding size may count as none
    finally:
        G.close()
