"""GPU: the Siddon projector on volumes with voxels that are not finite, bit for
bit against the oracle's per-ray traversal (both NaN or equal): a voxel that a
ray does not cross takes no part in its sum.
"""
import numpy as np
import pytest
import torch

from oracle_ffi import Geometry, Oracle
from test_gpu_parity import dev, to_desc
from tomogpi_amd import lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags", [0, lib.FLAG_INDEX_READS])
@pytest.mark.parametrize("dt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("where", ["corner", "outside", "inside"])
def test_siddon_nonfinite(ctx, where, dt, flags):
    """corner: voxel (0, 0, 0), outside the round field of view; outside: every voxel
    off the field of view and, in the end slices, off the rays; inside: a few."""
    g = Geometry(fod=90.0, fdd=180.0, nphi=12, su=40 * 2.0, sv=30 * 1.6, nu=40, nv=30, sx=36.0, sy=36.0, sz=28.0, nx=36,
                 ny=36, nz=28, num_start=1.0, den_start=7.0, num_stop=15.0, den_stop=8.0)
    print(f"[case] {where} {dt} flags={flags}", flush=True)
    o = Oracle(g)
    rng = np.random.default_rng(4)
    v = dev(rng.random(g.vol_shape, dtype=np.float32))
    if dt != "f32":
        v = v.to(torch.bfloat16 if dt == "bf16" else torch.float16)
    if where == "corner":
        v[0, 0, 0] = np.nan
    elif where == "outside":
        off = torch.from_numpy(o.siddon_T(np.ones(g.sino_shape)) == 0.0).cuda()
        v[off] = np.inf
    else:
        v[14, 18, 17] = np.inf
        v[20, 9, 25] = np.nan
    ref = o.siddon(v.float().cpu().numpy())
    assert np.isfinite(ref).sum() > 0.5 * ref.size
    G = lib.Geometry(ctx, to_desc(g))
    try:
        out = torch.zeros(g.sino_shape, dtype=torch.float32, device="cuda")
        G.project(v, out, lib.PROJ_SIDDON, flags)
        got = out.cpu().numpy()
        assert np.array_equal(got, ref, equal_nan=True), (np.isnan(got).sum(), np.isnan(ref).sum())
    finally:
        G.close()
