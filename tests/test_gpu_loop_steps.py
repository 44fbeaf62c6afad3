"""GPU: the loops' fused passes and device-side step rule against the same
iterations composed of the operators, norms and element-wise steps, bit for bit:
every sum keeps its order and every operation its rounding.
"""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle_ffi import Geometry
from test_gpu_parity import dev, to_desc
from tomogpi_amd import lib

pytestmark = pytest.mark.gpu


def _geom(n, nz, nphi):
    return Geometry(fod=2.0 * n, fdd=4.0 * n, nphi=nphi, su=2.0 * n, sv=2.0 * nz, nu=n, nv=nz, sx=float(n), sy=float(n),
                    sz=float(nz), nx=n, ny=n, nz=nz, num_start=1.0, den_start=7.0, num_stop=15.0, den_stop=8.0)


def _laplacian(x):
    z = torch.nn.functional.pad(x, (1, 1, 1, 1, 1, 1))
    c2 = x + x
    h = (c2 - z[1:-1, 1:-1, :-2]) - z[1:-1, 1:-1, 2:]
    v = (c2 - z[1:-1, :-2, 1:-1]) - z[1:-1, 2:, 1:-1]
    p = (c2 - z[:-2, 1:-1, 1:-1]) - z[2:, 1:-1, 1:-1]
    return (h + v) + p


def _f32(v):
    return float(np.float32(v))


def _compose(ctx, G, g, y, x, lam, iters, kopt, conjugate, weight):
    est, back = torch.empty_like(y), torch.empty_like(x)
    d, state, stats = None, -0.5, []
    for k in range(1, iters + 1):
        st = dict(residual_sq=0.0, norm_dj=0.0, norm_dj_proj=0.0, alpha=0.0, j_reg=0.0, beta=0.0)
        G.project(x, est, lib.PROJ_SIDDON)
        r = y - est
        st["residual_sq"] = lib.sq_norm(ctx, r)
        G.backproject(r * weight if weight is not None else r, back)
        gr = back * -2.0
        if lam != 0.0:
            lx = _laplacian(x)
            st["j_reg"] = lib.sq_norm(ctx, lx)
            gr = gr + _laplacian(lx) * _f32(2.0 * _f32(lam))
        if conjugate:
            gg = lib.sq_norm(ctx, gr)
            if k > 1:
                st["beta"] = gg / state
                d = d * _f32(st["beta"]) + gr
            else:
                d = gr
            state, top = gg, lib.dot(ctx, gr, d)
            st["norm_dj"] = gg
        else:
            d = gr
        if conjugate or k < kopt:
            if not conjugate:
                st["norm_dj"] = top = lib.sq_norm(ctx, d)
            G.project(d, est, lib.PROJ_SIDDON)
            reg = 2.0 * lib.sq_norm(ctx, _laplacian(d)) if lam != 0.0 else 0.0
            st["norm_dj_proj"] = 2.0 * lib.sq_norm(ctx, est) + lam * reg
            st["alpha"] = -top / st["norm_dj_proj"]
            if not conjugate:
                state = max(st["alpha"], state)
        else:
            st["alpha"] = state
        x = x + d * _f32(st["alpha"])
        stats.append(st)
    return x, stats


@pytest.mark.parametrize("form", ["gd", "cg", "wgd"])
@pytest.mark.parametrize("lam", [0.0, 0.03])
@pytest.mark.parametrize("n,nz,nphi", [(12, 9, 5), (91, 90, 70)])  # below and above 2048 blocks of 256 elements
def test_loop_steps(ctx, n, nz, nphi, lam, form):
    g = _geom(n, nz, nphi)
    print(f"[case] {n} {nz} {nphi} {lam} {form}", flush=True)
    G = lib.Geometry(ctx, to_desc(g))
    try:
        rng = np.random.default_rng(n)
        y, x0 = dev(rng.random(g.sino_shape, dtype=np.float32)), dev(rng.random(g.vol_shape, dtype=np.float32))
        w = dev(rng.random(g.sino_shape, dtype=np.float32)) if form == "wgd" else None
        x = x0.clone()
        got = G.gd_run(y, x, pair=lib.PAIR_SIDDONVI, iters=4, kopt=3, lam=lam, alpha_min_init=-0.5,
                       conjugate=form == "cg", weight=w)
        ref_x, ref = _compose(ctx, G, g, y, x0, lam, 4, 3, form == "cg", w)
        assert torch.equal(x, ref_x)
        for a, b in zip(got, ref):
            a = a if isinstance(a, dict) else {f: getattr(a, f) for f in b}
            assert {f: a[f] for f in b} == b
    finally:
        G.close()


def test_loop_statistics_in_pieces(ctx):
    """More iterations than the device keeps statistics of, and none asked for."""
    g = _geom(8, 6, 4)
    G = lib.Geometry(ctx, to_desc(g))
    try:
        y = dev(np.random.default_rng(2).random(g.sino_shape, dtype=np.float32))
        x, short = torch.zeros(g.vol_shape, device="cuda"), torch.zeros(g.vol_shape, device="cuda")
        # a fixed step small enough to fall for good: every iteration's residual is its own
        kw = dict(pair=lib.PAIR_SIDDONVI, kopt=1, alpha_min_init=-1e-6)
        many = G.gd_run(y, x, iters=1030, **kw)
        few = G.gd_run(y, short, iters=5, **kw)
        res = [s["residual_sq"] if isinstance(s, dict) else s.residual_sq for s in many]
        assert res[:5] == [s["residual_sq"] if isinstance(s, dict) else s.residual_sq for s in few]
        assert all(a > b > 0.0 for a, b in zip(res, res[1:]))
        p = lib.GdParams(pair=lib.PAIR_SIDDONVI, gradient_iteration_nb=1030, optimal_step_iteration_nb=1,
                         alpha_min_init=-1e-6)
        z = torch.zeros(g.vol_shape, device="cuda")
        torch.cuda.synchronize()
        assert ctx.lib.tomo_gd_run(ctx.h, G.h, C.byref(p), C.c_void_p(y.data_ptr()), C.c_void_p(z.data_ptr()), None,
                                   C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        assert torch.equal(x, z)
        sirt = G.sirt_run(y, x, pair=lib.PAIR_SIDDONVI, iters=1030, relaxation=1e-3)
        assert sirt[:5] == G.sirt_run(y, short, pair=lib.PAIR_SIDDONVI, iters=5, relaxation=1e-3)
        assert all(a > b > 0.0 for a, b in zip(sirt, sirt[1:]))
    finally:
        G.close()
