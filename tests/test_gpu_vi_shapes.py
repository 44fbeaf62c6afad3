"""GPU: the backprojector's column lengths and copies at their edges, bit for bit
against the oracle (FP16, whose u-weights are rounded: against each other).

Columns of 4, 8 or 16 voxels are picked from the number of workgroups; 4 and 8
stage 4 and 2 views between two barriers.  A box of taps is copied in 16-byte
pieces, by rows at the detector's ends, or not at all where it is too large.
"""
import numpy as np
import pytest
import torch

from oracle_ffi import Geometry, Oracle
from test_gpu_parity import dev, rel_l2, to_desc
from tomogpi_amd import lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("fdk", [False, True])
@pytest.mark.parametrize("nx,ny,nz,nu,nv,nphi,pixel,fod", [
    (33, 17, 9, 50, 20, 67, 2.0, 2.0), (64, 64, 64, 64, 64, 3, 2.0, 2.0), (40, 30, 3, 37, 5, 1, 2.0, 2.0),  # 4 voxels
    (64, 64, 64, 64, 64, 46, 2.0, 2.0),  # 4 voxels, boxes of up to 20 rows, the buffers' last, and two views left over
    (96, 90, 90, 150, 110, 66, 2.0, 2.0), (100, 100, 101, 101, 99, 7, 2.0, 2.0),                            # 8
    (137, 136, 130, 139, 133, 65, 2.0, 2.0), (130, 150, 150, 300, 200, 9, 2.0, 2.0),                        # 16
    (64, 64, 40, 200, 200, 6, 0.4, 2.0), (96, 96, 90, 400, 300, 5, 0.5, 2.0),  # boxes past the buffers
    (40, 40, 30, 24, 24, 21, 9.0, 2.0), (48, 40, 30, 1, 1, 5, 3.0, 2.0),       # many voxels a tap; one tap
    (40, 40, 200, 50, 5, 9, 2.0, 2.0), (90, 96, 260, 70, 9, 6, 2.0, 2.0),      # boxes more than 64 rows off the detector
    (64, 60, 50, 60, 50, 40, 2.0, 0.6),                                        # a source within the square
])
def test_vi_shapes(ctx, nx, ny, nz, nu, nv, nphi, pixel, fod, fdk, dt):
    print(f"[case] {nx} {ny} {nz} / {nu} {nv} {nphi} {pixel} {fod} {fdk} {dt}", flush=True)
    g = Geometry(fod=fod * nx, fdd=2.0 * fod * nx, nphi=nphi, su=nu * pixel, sv=nv * pixel, nu=nu, nv=nv, sx=float(nx),
                 sy=float(ny), sz=float(nz), nx=nx, ny=ny, nz=nz, num_start=1.0, den_start=7.0, num_stop=15.0,
                 den_stop=8.0)
    G = lib.Geometry(ctx, to_desc(g))
    try:
        s = dev(np.random.default_rng(nv).random(g.sino_shape, dtype=np.float32))
        s = s.to(torch.bfloat16) if dt == "bf16" else s
        o, host = Oracle(g), s.float().cpu().numpy()
        ref = o.vi_fdk(host) if fdk else o.vi(host)
        out = torch.full(g.vol_shape, np.nan, dtype=torch.float32, device="cuda")
        G.backproject(s, out, flags=lib.FLAG_FDK if fdk else 0)
        got = out.cpu().numpy()
        assert np.array_equal(got, ref), rel_l2(got, ref)
    finally:
        G.close()


@pytest.mark.parametrize("fdk", [False, True])
def test_vi_f16_column_lengths(ctx, fdk):
    """FP16 taps: the middle slices of volumes of 130, 66 and 20 slices (columns of
    16, 8 and 4 voxels) are the same bits."""
    nx, nu, nv, nphi = 136, 139, 133, 35
    s = dev(np.random.default_rng(1).random((nphi, nv, nu), dtype=np.float32)).to(torch.float16)
    mid = []
    for nz in (130, 66, 20):
        print(f"[case] {nx} {nz} / {nu} {nv} {nphi} {fdk}", flush=True)
        g = Geometry(fod=2.0 * nx, fdd=4.0 * nx, nphi=nphi, su=2.0 * nu, sv=2.0 * nv, nu=nu, nv=nv, sx=float(nx),
                     sy=float(nx), sz=float(nz), nx=nx, ny=nx, nz=nz, num_start=1.0, den_start=7.0, num_stop=15.0,
                     den_stop=8.0)
        G = lib.Geometry(ctx, to_desc(g))
        try:
            out = torch.full(g.vol_shape, np.nan, dtype=torch.float32, device="cuda")
            G.backproject(s, out, flags=lib.FLAG_FDK if fdk else 0)
            mid.append(out[nz // 2 - 10:nz // 2 + 10].cpu())
        finally:
            G.close()
    assert torch.equal(mid[0], mid[1]) and torch.equal(mid[0], mid[2])
