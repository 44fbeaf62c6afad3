"""GPU: VI whose box table or u-pair copy is made by more work items than one grid
dimension takes (2^24 workgroups).  The views that the launch reaches last hold the
only values."""
import numpy as np
import pytest
import torch

from oracle_ffi import Geometry, Oracle
from test_gpu_parity import rel_l2, to_desc
from tomogpi_amd import lib

pytestmark = pytest.mark.gpu


def _geom(n, nz, nu, nv, nphi, pixel):
    return Geometry(fod=2.0 * n, fdd=4.0 * n, nphi=nphi, su=nu * pixel, sv=nv * pixel, nu=nu, nv=nv, sx=float(n), sy=float(n),
                    sz=float(nz), nx=n, ny=n, nz=nz, num_start=0.0, den_start=1.0, num_stop=2.0, den_stop=1.0)


def _one_view(g, o, p, view):
    """delta times the bilinear reads of view p at the projections of the voxels, FP64."""
    i = o.info
    kw = dict(dtype=torch.float64, device="cuda")
    x = (torch.arange(g.nx, **kw) - i["cx"]).view(1, 1, -1)
    y = (torch.arange(g.ny, **kw) - i["cy"]).view(1, -1, 1)
    z = (torch.arange(g.nz, **kw) - i["cz"]).view(-1, 1, 1)
    ca, sa = np.cos(o.phi[p]), np.sin(o.phi[p])
    w = i["delta"] * (ca * x + sa * y) + g.fod
    u = g.fdd / i["du"] * i["delta"] * (ca * y - sa * x) / w + i["cu"] + 0.0 * z
    v = g.fdd / i["dv"] * i["delta"] * z / w + i["cv"]
    out = torch.zeros(g.vol_shape, **kw)
    pad = torch.nn.functional.pad(view.double(), (1, 1, 1, 1))
    uf, vf = torch.floor(u), torch.floor(v)
    for a in (0, 1):
        for b in (0, 1):
            wt = (u - uf if a else 1 - (u - uf)) * (v - vf if b else 1 - (v - vf))
            uu, vv = (uf + a + 1).clamp(0, g.nu + 1).long(), (vf + b + 1).clamp(0, g.nv + 1).long()
            out += wt * pad[vv, uu]
    return out * i["delta"]


def test_vi_many_boxes(ctx):
    """Rel-L2 <= 1e-5: u is rounded to FP32 below 64, 2^-18 of a weight."""
    g = _geom(2048, 1, 64, 2, 1030, 70.0)
    assert (g.nx // 32) * (g.ny // 8) * g.nphi > 1 << 24
    print("[case] boxes", flush=True)
    G, o = lib.Geometry(ctx, to_desc(g)), Oracle(g)
    try:
        y = torch.zeros(g.sino_shape, device="cuda")
        y[-3:] = torch.rand((3, g.nv, g.nu), device="cuda")
        out = torch.empty(g.vol_shape, device="cuda")
        G.backproject(y, out)
        ref = sum(_one_view(g, o, p, y[p]) for p in range(g.nphi - 3, g.nphi))
        assert rel_l2(out.cpu().numpy(), ref.cpu().numpy()) <= 1e-5
    finally:
        G.close()


def test_vi_many_pair_rows(ctx):
    """FP16 u-pairs of 2^24 rows and more; rel-L2 <= 1e-3, two steps of the FP16 u-weights."""
    g = _geom(16, 16, 32, 4096, 4100, 1.0)
    g.sv = 64.0
    print("[case] pairs", flush=True)
    G, o = lib.Geometry(ctx, to_desc(g)), Oracle(g)
    try:
        y = torch.zeros(g.sino_shape, dtype=torch.float16, device="cuda")
        y[-3:] = torch.rand((3, g.nv, g.nu), device="cuda").half()
        out = torch.empty(g.vol_shape, device="cuda")
        G.backproject(y, out)
        ref = sum(_one_view(g, o, p, y[p]) for p in range(g.nphi - 3, g.nphi))
        assert rel_l2(out.cpu().numpy(), ref.cpu().numpy()) <= 1e-3
    finally:
        G.close()
