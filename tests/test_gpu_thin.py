"""GPU: problems of few detector rows or few slices.  The projectors copy only the
planes that rays reach and pick waves of few rows: bit for bit against the oracle.
"""
import numpy as np
import pytest
import torch

from oracle_ffi import Geometry, Oracle
from test_gpu_parity import dev, rel_l2, to_desc
from tomogpi_amd import lib

pytestmark = pytest.mark.gpu


def _geom(nx, ny, nz, nu, nv, nphi, pixel=2.0, fod=2.5, fdd=2.0):
    return Geometry(fod=fod * nx, fdd=fdd * fod * nx, nphi=nphi, su=nu * 2.0, sv=nv * pixel, nu=nu, nv=nv, sx=float(nx),
                    sy=float(ny), sz=float(nz), nx=nx, ny=ny, nz=nz, num_start=1.0, den_start=7.0, num_stop=15.0,
                    den_stop=8.0)


@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("nx,ny,nz,nu,nv,nphi,pixel,fod", [
    (37, 33, 90, 41, 1, 5, 2.0, 2.5), (36, 36, 91, 70, 2, 6, 2.0, 2.5), (37, 33, 120, 40, 3, 4, 1.0, 2.5),  # few rows, many planes
    (33, 37, 70, 30, 8, 5, 2.0, 2.5), (33, 33, 150, 66, 20, 5, 2.5, 0.8), (36, 12, 64, 40, 6, 8, 3.0, 1.2),
    (37, 33, 8, 41, 4, 5, 2.0, 2.5), (36, 36, 9, 70, 5, 6, 1.5, 2.5),      # reach near the volume's height
    (37, 33, 1, 41, 64, 5, 2.0, 2.5), (36, 36, 4, 70, 90, 6, 2.0, 2.5), (33, 37, 16, 35, 33, 4, 2.0, 0.9),  # few slices
])
def test_thin_projections(ctx, nx, ny, nz, nu, nv, nphi, pixel, fod, dt):
    g = _geom(nx, ny, nz, nu, nv, nphi, pixel, fod)
    print(f"[case] {nx} {ny} {nz} / {nu} {nv} {nphi} {dt}", flush=True)
    G, o = lib.Geometry(ctx, to_desc(g)), Oracle(g)
    try:
        v = dev(np.random.default_rng(nv).random(g.vol_shape, dtype=np.float32))
        if dt != "f32":
            v = v.to(torch.bfloat16 if dt == "bf16" else torch.float16)
        vol = v.float().cpu().numpy()
        for op, cube, ref in (("siddon", 0, o.siddon(vol)), ("rs", 0, o.rs(vol)), ("rs", 1, o.rs(vol, cube=True))):
            for extra in (0, lib.FLAG_INDEX_READS):
                out = torch.full(g.sino_shape, np.nan, dtype=torch.float32, device="cuda")
                G.project(v, out, lib.PROJ_SIDDON if op == "siddon" else lib.PROJ_RS,
                          extra | (lib.FLAG_RS_FOV_CUBE if cube else 0))
                got = out.cpu().numpy()
                assert np.array_equal(got, ref), (op, cube, extra, rel_l2(got, ref))
    finally:
        G.close()


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("ny,nz,nu,nv,nphi", [
    (24, 1, 300, 1, 260), (20, 60, 300, 1, 260),     # a row a wave
    (24, 2, 300, 2, 260), (24, 40, 260, 2, 130), (24, 2, 260, 64, 130),  # two
    (24, 3, 290, 3, 130), (24, 5, 260, 6, 130), (24, 8, 260, 9, 130),    # four, eight
    (24, 14, 200, 20, 90), (24, 6, 260, 70, 90), (24, 30, 130, 37, 60),  # and more; rows off the volume
])
def test_thin_wave_rows(ctx, ny, nz, nu, nv, nphi, dt):
    """Enough rays for waves of few rows."""
    g = _geom(24, ny, nz, nu, nv, nphi, fod=1.953125)
    g.su = nu * 0.25
    print(f"[case] {ny} {nz} / {nu} {nv} {nphi} {dt}", flush=True)
    G, o = lib.Geometry(ctx, to_desc(g)), Oracle(g)
    try:
        v = dev(np.random.default_rng(nv).random(g.vol_shape, dtype=np.float32)).to(
            torch.float32 if dt == "f32" else torch.bfloat16)
        vol = v.float().cpu().numpy()
        for op, cube, ref in (("siddon", 0, o.siddon(vol)), ("rs", 0, o.rs(vol)), ("rs", 1, o.rs(vol, cube=True))):
            for extra in (0, lib.FLAG_INDEX_READS):
                out = torch.full(g.sino_shape, np.nan, dtype=torch.float32, device="cuda")
                G.project(v, out, lib.PROJ_SIDDON if op == "siddon" else lib.PROJ_RS,
                          extra | (lib.FLAG_RS_FOV_CUBE if cube else 0))
                got = out.cpu().numpy()
                assert np.array_equal(got, ref), (op, cube, extra, rel_l2(got, ref))
    finally:
        G.close()


@pytest.mark.parametrize("pair", [lib.PAIR_SIDDONVI, lib.PAIR_RSVI])
def test_thin_loop_and_server(ctx, pair):
    """A loop and a served request of few rows over many planes, in FP32 as the
    oracle's loop (rel-L2 1e-6, the bound of the loops' parity tests), and both
    through BF16 copies (2e-2: nine operators whose inputs are rounded at 2^-9)."""
    g = _geom(36, 36, 80, 40, 5, 12)
    print(f"[case] pair={pair}", flush=True)
    y = np.random.default_rng(3).random(g.sino_shape, dtype=np.float32)
    kw = dict(iters=3, kopt=4, lam=0.01)
    ref, _ = Oracle(g).gd(y, pair=pair, **kw)
    G, srv = lib.Geometry(ctx, to_desc(g)), lib.Server(ctx, max_active=4)
    try:
        for storage, bound in ((lib.F32, 1e-6), (lib.BF16, 2e-2)):
            x, z = torch.zeros(g.vol_shape, device="cuda"), torch.empty(g.vol_shape, device="cuda")
            G.gd_run(dev(y), x, pair=pair, storage=storage, **kw)
            assert rel_l2(x.cpu().numpy(), ref) <= bound
            d = dev(y)
            torch.cuda.synchronize()
            srv.wait(srv.submit(to_desc(g), d, z, pair=pair, storage=storage, **kw))
            torch.cuda.synchronize()
            assert rel_l2(z.cpu().numpy(), ref) <= bound
    finally:
        srv.close()
        G.close()


@pytest.mark.parametrize("pair", [lib.PAIR_SIDDONVI, lib.PAIR_RSVI])
def test_thin_server_rows(ctx, pair):
    """Served requests whose waves hold few rows, two of different shapes at once
    (rel-L2 1e-6, the bound of the served results)."""
    kw = dict(iters=2, kopt=3, lam=0.01)
    print(f"[case] pair={pair}", flush=True)
    srv, jobs = lib.Server(ctx, max_active=4), []
    try:
        for nz, nu, nv, nphi in ((6, 260, 6, 130), (1, 300, 1, 260)):
            g = _geom(24, 24, nz, nu, nv, nphi, fod=1.953125)
            g.su = nu * 0.25
            y = np.random.default_rng(nv).random(g.sino_shape, dtype=np.float32)
            jobs.append((g, y, dev(y), torch.empty(g.vol_shape, device="cuda")))
        torch.cuda.synchronize()
        ids = [srv.submit(to_desc(g), d, z, pair=pair, **kw) for g, _, d, z in jobs]
        for i in ids:
            srv.wait(i)
        torch.cuda.synchronize()
        for g, y, _, z in jobs:
            ref, _ = Oracle(g).gd(y, pair=pair, **kw)
            assert rel_l2(z.cpu().numpy(), ref) <= 1e-6
    finally:
        srv.close()
