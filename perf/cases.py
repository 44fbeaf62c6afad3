"""Performance cases of the cone-beam operators and the loops that call them.

Every case is one call that a user's program makes through the public Python
interface (tomogpi_amd.lib): a projection, a backprojection, an exact
transpose, a reconstruction loop or a batch of served reconstructions.
Volumes are sums of random ellipsoids and sinograms their analytic cone-beam
projections, made from the seed with torch alone.

A case is a dict of plain values:
  op      siddon, rs, vi, fdk           projections and backprojections
          siddon_t, rs_t, vi_t          exact transposes
          gd, cg, sirt                  reconstruction loops
          serve                         several reconstructions through a server
  nx, ny, nz, nu, nv, views, pixel      the acquisition (1 mm voxels, pixel in mm)
  start, stop                           angular range in units of pi
  dtype   f32, f16, bf16                element type of both operands (transposes
                                        write f32; loops: type of the operators' inputs)
  pair, iters, cube                     loops' operator pair and iterations, RS field of view
"""
import math

import numpy as np
import torch

from tomogpi_amd import lib

DEVICE = "cuda"
FORWARD = ("siddon", "rs", "vi_t")            # volume -> sinogram
LOOPS = ("gd", "cg", "sirt")
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
LAMBDA = 0.01
EXACT_MOST = 1.0e10                           # voxel-view updates the 64-bit forms are evaluated for


def _case(name, op, n, views, nu=None, nv=None, pixel=2.0, dtype="f32", pair="siddonvi", iters=0, cube=False,
          start=0.0, stop=2.0):
    nx, ny, nz = (n, n, n) if isinstance(n, int) else n
    c = dict(op=op, nx=nx, ny=ny, nz=nz, nu=nu or nx, nv=nv or nz, views=views, pixel=pixel, start=start, stop=stop,
             dtype=dtype, pair=pair, iters=iters, cube=cube)
    return dict(c, name=name) if name else c


def listed():
    return [
        # The smallest calls: one operator of a 64^3 volume, as in a coarse level
        # or a parameter scan, where launches and latency count.
        _case("siddon_64", "siddon", 64, 48),
        _case("vi_64", "vi", 64, 48),
        # A whole regularised reconstruction of the size most served requests have.
        _case("gd_128", "gd", 128, 180, iters=5),
        # The 256^3 / 256-view acquisition of the shipped configuration.
        _case("rs_256", "rs", 256, 256),
        # FDK, the one-pass reconstruction, of that volume from 360 views.
        _case("fdk_256", "fdk", 256, 360),
        # The transpose of the projector, for solvers that need the exact adjoint.
        _case("siddon_t_256", "siddon_t", 256, 256),
        # The transpose of the backprojector on a short scan with odd sizes.
        _case("vi_t_odd", "vi_t", (201, 187, 149), 131, nu=229, nv=173, stop=1.25),
        # 16-bit storage with odd sizes and a detector that is not square.
        _case("rs_f16_odd", "rs", (387, 365, 291), 211, nu=401, nv=307, dtype="f16"),
        # The workload the benchmark quotes: 512^3, 512 views, both directions.
        _case("siddon_512", "siddon", 512, 512),
        _case("vi_512", "vi", 512, 512),
        # The largest acquisition of the benchmark: 1024^3, 720 views, 768 x 512 cells.
        _case("siddon_1024", "siddon", 1024, 720, nu=768, nv=512, pixel=4.0),
        # Uneven requests at one server, as a reconstruction service has them.
        _case("serve_mix", "serve", 128, 90, iters=4),
    ]


def draw(rng):
    op = rng.choice(["siddon", "siddon", "rs", "rs", "vi", "vi", "fdk", "siddon_t", "rs_t", "vi_t", "gd", "cg",
                     "sirt", "serve"])
    if op == "serve":
        return _case(None, op, int(40 * 3.5 ** rng.random()), rng.randint(24, 100), iters=rng.randint(2, 4))
    top = 160 if op in LOOPS else 272 if op.endswith("_t") else 512
    n = int(round(24 * (top / 24.0) ** rng.random()))
    if rng.random() < 0.5:
        shape = tuple(max(17, int(n * rng.uniform(0.7, 1.0))) for _ in range(3))
    else:
        shape = (n, n, n)
    pixel = rng.choice([2.0, 2.0, 1.6, 2.4])
    nu = max(17, int(shape[0] * rng.uniform(0.8, 1.4))) if rng.random() < 0.5 else shape[0]
    nv = max(17, int(shape[2] * rng.uniform(0.8, 1.3))) if rng.random() < 0.5 else shape[2]
    if nu % 2 and (shape[0] % 2 == 0 or shape[1] % 2 == 0):
        nu += 1  # else the middle column's rays run along a plane between voxels in some views: two right answers
    views = int(round(16 * (max(32, min(360, n)) / 16.0) ** rng.random()))
    if op in LOOPS:
        dtype = rng.choice(["f32", "f32", "f16", "bf16"]) if op != "sirt" else "f32"
        return _case(None, op, shape, min(views, 180), nu, nv, pixel, dtype, rng.choice(["siddonvi", "rsvi"]),
                     rng.randint(2, 5))
    return _case(None, op, shape, views, nu, nv, pixel, rng.choice(["f32", "f32", "f16", "bf16"]),
                 cube=op.startswith("rs") and rng.random() < 0.4, start=rng.choice([0.0, 0.0, 0.25]),
                 stop=rng.choice([2.0, 2.0, 1.25]))


# ---- the acquisition ------------------------------------------------------------
class _Geometry:
    """The acquisition in plain numbers (float-typed sizes as the interface has them)."""

    def __init__(self, c):
        self.nx, self.ny, self.nz, self.nu, self.nv, self.views = (c[k] for k in ("nx", "ny", "nz", "nu", "nv", "views"))
        k = self.nx / 256.0
        self.fod, self.fdd = 500.0 * k, 1000.0 * k
        f = np.float32
        self.su, self.sv = float(f(self.nu * c["pixel"])), float(f(self.nv * c["pixel"]))
        self.du, self.dv = float(f(self.su) / f(self.nu)), float(f(self.sv) / f(self.nv))
        self.delta = 1.0
        self.cu, self.cv = self.nu / 2 - 0.5, self.nv / 2 - 0.5
        self.cx, self.cy, self.cz = self.nx / 2 - 0.5, self.ny / 2 - 0.5, self.nz / 2 - 0.5
        self.start, self.stop = c["start"], c["stop"]
        step = math.pi * (self.stop - self.start) / self.views
        self.phi = [(p + self.start) * step for p in range(self.views)]
        self.updates = float(self.nx) * self.ny * self.nz * self.views

    def desc(self):
        return lib.AcquisitionDesc(
            fod_mm=self.fod, fdd_mm=self.fdd, projection_nb=self.views, u_detector_size_mm=self.su,
            v_detector_size_mm=self.sv, u_pixel_nb=self.nu, v_pixel_nb=self.nv, x_volume_size_mm=float(self.nx),
            y_volume_size_mm=float(self.ny), z_volume_size_mm=float(self.nz), x_pixel_nb=self.nx, y_pixel_nb=self.ny,
            z_pixel_nb=self.nz, num_start_angle=self.start, den_start_angle=1.0, num_stop_angle=self.stop,
            den_stop_angle=1.0)

    def rays(self, p0, p1, dtype=torch.float64):
        """Source (x, y) and unit directions of the cells of views p0 .. p1 - 1, mm."""
        kw = dict(dtype=dtype, device=DEVICE)
        phi = torch.tensor(self.phi[p0:p1], dtype=torch.float64)
        ca, sa = torch.cos(phi).to(**kw).view(-1, 1, 1), torch.sin(phi).to(**kw).view(-1, 1, 1)
        s = ((torch.arange(self.nu, **kw) - self.cu) * self.du).view(1, 1, -1)
        t = ((torch.arange(self.nv, **kw) - self.cv) * self.dv).view(1, -1, 1)
        rx, ry, rz = ca * self.fdd - s * sa, sa * self.fdd + s * ca, t
        length = torch.sqrt(rx * rx + ry * ry + rz * rz)
        one = torch.ones_like(length)
        return [(-self.fod * ca) * one, (-self.fod * sa) * one, torch.zeros_like(length)], [rx / length, ry / length,
                                                                                           rz / length]


def _parts(c):
    """The reconstructions of a served batch: sizes of the case's and smaller."""
    out = []
    for i, f in enumerate((1.0, 0.5, 0.75, 0.5, 1.25, 0.6)):
        n = max(24, int(c["nx"] * f))
        out.append(dict(c, op="gd", nx=n, ny=n, nz=n, nu=n, nv=n, pair=("rsvi", "siddonvi")[i % 2]))
    return out


# ---- inputs ---------------------------------------------------------------------
def _ellipsoids(g, seed, count=24):
    """Rows (centre, semi-axis-scaled rotation, density) of random ellipsoids in the inner 80%, mm from the centre."""
    r = np.random.RandomState(seed % (1 << 31))
    size = np.array([g.nx, g.ny, g.nz], dtype=np.float64)
    out = []
    for _ in range(count):
        q = r.normal(size=4)
        w, x, y, z = q / np.linalg.norm(q)
        rot = np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)],
                        [2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)],
                        [2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]])
        semi = r.uniform(0.01, 0.23, 3) * size.min() + 1.0
        out.append(((r.rand(3) - 0.5) * 0.8 * size, rot / semi[:, None], r.rand()))
    return out


def _volume(g, seed):
    kw = dict(dtype=torch.float32, device=DEVICE)
    vol = torch.zeros((g.nz, g.ny, g.nx), **kw)
    x = (torch.arange(g.nx, **kw) - g.cx).view(1, 1, -1)
    y = (torch.arange(g.ny, **kw) - g.cy).view(1, -1, 1)
    z = (torch.arange(g.nz, **kw) - g.cz).view(-1, 1, 1)
    for c, m, rho in _ellipsoids(g, seed):
        # the slices and the box the ellipsoid can reach
        reach = 1.0 / np.linalg.norm(m, axis=1).min()
        lo = [max(0, int(v - reach + o)) for v, o in zip(c, (g.cx, g.cy, g.cz))]
        hi = [min(n, int(v + reach + o) + 2) for v, o, n in zip(c, (g.cx, g.cy, g.cz), (g.nx, g.ny, g.nz))]
        if any(h <= l for l, h in zip(lo, hi)):
            continue
        dx, dy = x[..., lo[0]:hi[0]] - c[0], y[:, lo[1]:hi[1]] - c[1]
        for z0 in range(lo[2], hi[2], 64):
            z1 = min(z0 + 64, hi[2])
            dz = z[z0:z1] - c[2]
            q = sum((float(r[0]) * dx + float(r[1]) * dy + float(r[2]) * dz) ** 2 for r in m)
            vol[z0:z1, lo[1]:hi[1], lo[0]:hi[0]] += (q <= 1.0) * float(rho)
    return vol


def _sinogram(g, seed):
    """Chords through the ellipsoids times their densities, mm."""
    sino = torch.empty((g.views, g.nv, g.nu), dtype=torch.float32, device=DEVICE)
    table = _ellipsoids(g, seed)
    step = max(1, (1 << 25) // (g.nu * g.nv))
    for p in range(0, g.views, step):
        src, d = g.rays(p, min(g.views, p + step), torch.float32)
        acc = torch.zeros_like(d[0])
        for c, m, rho in table:
            o = [src[k] - float(c[k]) for k in range(3)]
            e = [sum(float(r[k]) * o[k] for k in range(3)) for r in m]
            f = [sum(float(r[k]) * d[k] for k in range(3)) for r in m]
            a, b = sum(v * v for v in f), sum(u * v for u, v in zip(e, f))
            # squared distance of the ray from the centre, in semi-axes
            miss = sum((u - b / a * v) ** 2 for u, v in zip(e, f))
            acc += 2.0 * float(rho) * torch.sqrt(torch.clamp((1.0 - miss) / a, min=0.0))
        sino[p:p + step] = acc
    return sino


def _power(limit, top):
    return 2.0 ** math.floor(math.log2(limit / top)) if top > 0 else 1.0


def _data(c, seed):
    """(geometry, input as stored, its scale, scale of the result) of an operator case."""
    g = _Geometry(c)
    x = _volume(g, seed) if c["op"] in FORWARD else _sinogram(g, seed)
    scale = out_scale = 1.0
    if c["dtype"] == "f16":
        top = float(x.abs().max())
        scale = _power(16384.0, top)
        # no sum of the path exceeds the longest chord (projections) or the views (backprojections) times the largest value
        reach = 1.5 * max(g.nx, g.ny, g.nz) if c["op"] in FORWARD else float(g.views)
        out_scale = 1.0 if c["op"].endswith("_t") else _power(32768.0, max(top, 1e-6) * reach)
    x = (x * scale).to(DTYPES[c["dtype"]]) if c["dtype"] != "f32" else x
    return g, x, scale, out_scale


_context = []


def _ctx():
    if not _context:
        _context.append(lib.Context(0))
    return _context[0]


def prepare(case, seed):
    c = case
    if c["op"] == "serve":
        parts = _parts(c)
        geoms = [_Geometry(p) for p in parts]
        sinos = [_sinogram(g, seed + 101 * i) for i, g in enumerate(geoms)]
        vols = [torch.empty((g.nz, g.ny, g.nx), dtype=torch.float32, device=DEVICE) for g in geoms]
        return dict(case=c, parts=parts, descs=[g.desc() for g in geoms], sinos=sinos, vols=vols,
                    server=lib.Server(_ctx(), max_active=8))
    if c["op"] in LOOPS:
        g = _Geometry(c)
        return dict(case=c, geom=lib.Geometry(_ctx(), g.desc()), sino=_sinogram(g, seed),
                    vol=torch.empty((g.nz, g.ny, g.nx), dtype=torch.float32, device=DEVICE))
    g, x, scale, out_scale = _data(c, seed)
    shape = (g.views, g.nv, g.nu) if c["op"] in FORWARD else (g.nz, g.ny, g.nx)
    kind = torch.float32 if c["op"].endswith("_t") else DTYPES[c["dtype"]]
    return dict(case=c, geom=lib.Geometry(_ctx(), g.desc()), x=x, scale=scale, out_scale=out_scale,
                out=torch.empty(shape, dtype=kind, device=DEVICE))


_PAIR = {"rsvi": lib.PAIR_RSVI, "siddonvi": lib.PAIR_SIDDONVI}
_STORAGE = {"f32": lib.F32, "f16": lib.F16, "bf16": lib.BF16}


def run(state):
    c = state["case"]
    op = c["op"]
    if op == "serve":
        torch.cuda.current_stream().synchronize()  # the server reads the inputs on its own stream
        srv = state["server"]
        ids = [srv.submit(d, s, v, pair=_PAIR[p["pair"]], iters=p["iters"], kopt=p["iters"] + 1, lam=LAMBDA)
               for p, d, s, v in zip(state["parts"], state["descs"], state["sinos"], state["vols"])]
        for i in ids:
            srv.wait(i)
        return state["vols"]
    g = state["geom"]
    if op in LOOPS:
        vol = state["vol"]
        if op == "sirt":
            res = g.sirt_run(state["sino"], vol, pair=_PAIR[c["pair"]], iters=c["iters"])
        else:
            vol.zero_()
            st = g.gd_run(state["sino"], vol, pair=_PAIR[c["pair"]], iters=c["iters"], kopt=c["iters"] + 1, lam=LAMBDA,
                          conjugate=op == "cg", storage=_STORAGE[c["dtype"]])
            res = [s["residual_sq"] for s in st]
        return {"volume": vol, "residual": np.array(res, dtype=np.float32)}
    x, out, si, so = state["x"], state["out"], state["scale"], state["out_scale"]
    cube = lib.FLAG_RS_FOV_CUBE if c["cube"] else 0
    if op == "siddon":
        return g.project(x, out, lib.PROJ_SIDDON, vol_scale=si, sino_scale=so)
    if op == "rs":
        return g.project(x, out, lib.PROJ_RS, cube, vol_scale=si, sino_scale=so)
    if op in ("vi", "fdk"):
        return g.backproject(x, out, flags=lib.FLAG_FDK if op == "fdk" else 0, sino_scale=si, vol_scale=so)
    if op == "vi_t":
        return g.backproject_adjoint(x, out, vol_scale=si)
    return g.project_adjoint(x, out, lib.PROJ_RS if op == "rs_t" else lib.PROJ_SIDDON, cube, sino_scale=si)


# ---- work -----------------------------------------------------------------------
def work(case):
    """Bytes: volume and sinogram once each.  Flops: three chords a slab and ray
    (Siddon, 2 each), seven lerps and the sum per sample (RS, 22), three lerps
    and the sum per voxel and view (VI, 10)."""
    c = case
    if c["op"] == "serve":
        each = [work(p) for p in _parts(c)]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    g = _Geometry(c)
    vox, cells = float(g.nx) * g.ny * g.nz, float(g.nu) * g.nv * g.views
    siddon, rs, vi = cells * 0.8 * g.nx * 6.0, cells * 0.8 * g.nx * 22.0, g.updates * 10.0
    if c["op"] in LOOPS:
        proj = siddon if c["pair"] == "siddonvi" else rs
        projections = 1 if c["op"] == "sirt" else 2
        return {"bytes": 4.0 * (vox + cells), "flops": c["iters"] * (projections * proj + vi)}
    size = 4 if c["dtype"] == "f32" else 2
    out = 4 if c["op"].endswith("_t") else size
    n_in, n_out = (vox, cells) if c["op"] in FORWARD else (cells, vox)
    return {"bytes": size * n_in + out * n_out,
            "flops": {"s": siddon, "r": rs, "v": vi, "f": vi * 1.6}[c["op"][0]]}


# ---- 64-bit results ---------------------------------------------------------------
def _chunks(g, cells):
    step = max(1, cells // (g.nu * g.nv))
    return [(p, min(g.views, p + step)) for p in range(0, g.views, step)]


def _circle(src, d, radius2):
    a = d[0] * d[0] + d[1] * d[1]
    b = src[0] * d[0] + src[1] * d[1]
    disc = b * b - a * (src[0] * src[0] + src[1] * src[1] - radius2)
    ok = disc > 0.0
    root = torch.sqrt(torch.clamp(disc, min=0.0))
    return ok, (-b - root) / a, (-b + root) / a


def _siddon64(g, vol, sino=None):
    """Chord sums through the inscribed cylinder cut by the volume's z extent;
    with `sino`, the transpose: its values times the chords, added to a volume.
    Where the cylinder is wider than the grid, the stretch before the grid
    counts for the border voxel it leads to and the one after it for none."""
    out = torch.zeros((g.views, g.nv, g.nu) if sino is None else (g.nz * g.ny * g.nx,), dtype=torch.float64,
                      device=DEVICE)
    flat = vol.reshape(-1) if sino is None else None
    n = (g.nx, g.ny, g.nz)
    cen = (g.cx, g.cy, g.cz)
    stride = (1, g.nx, g.nx * g.ny)
    for p0, p1 in _chunks(g, 1 << 22):
        src, d = g.rays(p0, p1)
        ok, l0, l1 = _circle(src, d, (0.5 * g.nx) ** 2)
        far = torch.full_like(l0, 1e30)
        dz = torch.where(d[2] == 0.0, torch.full_like(l0, 1e-300), d[2])
        za, zb = (-0.5 * g.nz) / dz, (0.5 * g.nz) / dz
        l0 = torch.where(d[2] == 0.0, l0, torch.maximum(l0, torch.minimum(za, zb)))
        l1 = torch.where(d[2] == 0.0, l1, torch.minimum(l1, torch.maximum(za, zb)))
        ok = ok & (l1 > l0)
        for ax in (0, 1):
            mine = ok & ((d[0].abs() >= d[1].abs()) if ax == 0 else (d[0].abs() < d[1].abs()))
            at = mine.reshape(-1).nonzero().squeeze(1)
            if at.numel() == 0:
                continue
            S = [v.reshape(-1)[at] for v in src]
            D = [v.reshape(-1)[at] for v in d]
            a, b = l0.reshape(-1)[at], l1.reshape(-1)[at]
            acc = torch.zeros_like(a)
            gv = sino[p0:p1].reshape(-1)[at] if sino is not None else None
            others = [k for k in range(3) if k != ax]
            beyond = max(0, (g.nx - n[ax]) // 2 + 1) if g.nx > n[ax] else 0
            for i in range(-beyond, n[ax] + beyond):
                # the slab's two planes, cut to the field of view
                e0, e1 = (i - 0.5 - cen[ax] - S[ax]) / D[ax], (i + 0.5 - cen[ax] - S[ax]) / D[ax]
                t0, t1 = torch.maximum(torch.minimum(e0, e1), a), torch.minimum(torch.maximum(e0, e1), b)
                cuts = []
                for k in others:
                    # the plane between voxels crossed inside the slab, if one is
                    x0, x1 = S[k] + t0 * D[k] + cen[k] + 0.5, S[k] + t1 * D[k] + cen[k] + 0.5
                    plane = torch.floor(torch.maximum(x0, x1))
                    t = (plane - 0.5 - cen[k] - S[k]) / torch.where(D[k] == 0.0, far.reshape(-1)[at], D[k])
                    cuts.append(torch.where((t > t0) & (t < t1) & (D[k] != 0.0), t, t1))
                c1, c2 = torch.minimum(*cuts), torch.maximum(*cuts)
                for u, v in ((t0, c1), (c1, c2), (c2, t1)):
                    chord, mid = v - u, 0.5 * (u + v)
                    o = torch.full_like(at, min(max(i, 0), n[ax] - 1) * stride[ax])
                    good = chord > 0.0
                    if i < 0 or i >= n[ax]:
                        good = good & ((D[ax] > 0.0) if i < 0 else (D[ax] < 0.0))
                    for k in others:
                        q = torch.floor(S[k] + mid * D[k] + cen[k] + 0.5)
                        good = good & ((q >= 0) | (D[k] > 0.0)) & ((q < n[k]) | (D[k] < 0.0))
                        o += q.clamp(0, n[k] - 1).long() * stride[k]
                    chord = torch.where(good, chord, torch.zeros_like(chord))
                    if sino is None:
                        acc += chord * flat[o]
                    else:
                        out.index_add_(0, o, chord * gv)
            if sino is None:
                out[p0:p1].reshape(-1)[at] = acc
    return out if sino is None else out.view(g.nz, g.ny, g.nx)


def _rs64(g, vol, cube, sino=None):
    """Trilinear samples one voxel apart from the entry, times the voxel size;
    with `sino`, the transpose."""
    out = torch.zeros((g.views, g.nv, g.nu) if sino is None else (g.nz * g.ny * g.nx,), dtype=torch.float64,
                      device=DEVICE)
    flat = vol.reshape(-1) if sino is None else None
    n = (g.nx, g.ny, g.nz)
    for p0, p1 in _chunks(g, 1 << 22):
        src, d = g.rays(p0, p1)
        ok, l1, l2 = _circle(src, d, (2.0 if cube else 1.0) * (0.5 * g.nx) ** 2)
        if cube:
            for k, m in ((0, g.nx), (1, g.ny)):
                lo, hi = -(m / 2 - 0.5), m / 2 - 0.5
                flatd = d[k] == 0.0
                dk = torch.where(flatd, torch.full_like(l1, 1e-300), d[k])
                ta, tb = (lo - src[k]) / dk, (hi - src[k]) / dk
                l1 = torch.where(flatd, l1, torch.maximum(l1, torch.minimum(ta, tb)))
                l2 = torch.where(flatd, l2, torch.minimum(l2, torch.maximum(ta, tb)))
                ok = ok & (~flatd | ((src[k] >= lo) & (src[k] <= hi)))
            ok = ok & (l1 <= l2)
        ze, zx = l1 * d[2] + g.cz, l2 * d[2] + g.cz
        ok = ok & (ze >= 0.0) & ((ze <= g.nz - 1) if cube else (ze < g.nz))
        dz = torch.where(d[2] == 0.0, torch.full_like(l1, 1e-300), d[2])
        l2 = torch.where(zx > g.nz - 1, (g.nz - 1 - g.cz) / dz, torch.where(zx < 0.0, -g.cz / dz, l2))
        count = torch.where(ok, torch.floor((l2 - l1).abs()), torch.zeros_like(l1))
        at = (count >= 1).reshape(-1).nonzero().squeeze(1)
        if at.numel() == 0:
            continue
        D = [v.reshape(-1)[at] for v in d]
        E = [(src[k] + l1 * d[k]).reshape(-1)[at] + c for k, c in enumerate((g.cx, g.cy, g.cz))]
        count = count.reshape(-1)[at]
        gv = sino[p0:p1].reshape(-1)[at] if sino is not None else None
        acc = torch.zeros_like(count)
        for s in range(int(count.max())):
            x = [E[k] + s * D[k] for k in range(3)]
            f = [torch.floor(v) for v in x]
            w = [v - u for v, u in zip(x, f)]
            live = count > s
            for corner in range(8):
                o, wt = torch.zeros_like(at), live.to(torch.float64)
                for k, stride in enumerate((1, g.nx, g.nx * g.ny)):
                    up = (corner >> k) & 1
                    q = f[k] + up
                    wt = wt * (w[k] if up else 1.0 - w[k]) * ((q >= 0) & (q < n[k]))
                    o += q.clamp(0, n[k] - 1).long() * stride
                if sino is None:
                    acc += wt * flat[o]
                else:
                    out.index_add_(0, o, wt * gv)
        if sino is None:
            out[p0:p1].reshape(-1)[at] = acc
    return out * g.delta if sino is None else (out * g.delta).view(g.nz, g.ny, g.nx)


def _vi64(g, sino, fdk=False, vol=None):
    """Bilinear reads of every view at the voxel's projection, summed times the
    voxel size (FDK: weighted); with `vol`, the transpose."""
    kw = dict(dtype=torch.float64, device=DEVICE)
    out = torch.zeros((g.nz, g.ny, g.nx) if vol is None else (g.views, g.nv * g.nu), **kw)
    x = (torch.arange(g.nx, **kw) - g.cx).view(1, -1)
    y = (torch.arange(g.ny, **kw) - g.cy).view(-1, 1)
    z = (torch.arange(g.nz, **kw) - g.cz).view(-1, 1, 1)
    ku, kv = g.fdd / g.du, g.fdd / g.dv
    for p, phi in enumerate(g.phi):
        ca, sa = math.cos(phi), math.sin(phi)
        w = ca * x + sa * y + g.fod
        u = ku * (-sa * x + ca * y) / w + g.cu
        slope = kv / w
        uf = torch.floor(u)
        fu = u - uf
        zs = max(1, (1 << 24) // (g.nx * g.ny))
        for z0 in range(0, g.nz, zs):
            v = z[z0:z0 + zs] * slope + g.cv
            vf = torch.floor(v)
            fv = v - vf
            part = 0.0
            for a in (0, 1):
                for b in (0, 1):
                    uu, vv = uf + a, vf + b
                    wt = (fu if a else 1.0 - fu) * (fv if b else 1.0 - fv) * (
                        (uu >= 0) & (uu < g.nu) & (vv >= 0) & (vv < g.nv))
                    o = vv.clamp(0, g.nv - 1).long() * g.nu + uu.clamp(0, g.nu - 1).long()
                    if vol is None:
                        part = part + wt * sino[p].reshape(-1)[o]
                    else:
                        out[p].index_add_(0, o.reshape(-1), (wt * vol[z0:z0 + zs]).reshape(-1))
            if vol is None:
                if fdk:
                    up, vp = u - g.cu, v - g.cv
                    alpha = math.pi * g.fod * g.fdd / g.views
                    part = part * (alpha * ku / (w * w)) / torch.sqrt(ku * ku + up * up + vp * vp)
                out[z0:z0 + zs] += part
    if vol is not None:
        return (out * g.delta).view(g.views, g.nv, g.nu)
    return out if fdk else out * g.delta


def _laplacian64(x):
    y = 6.0 * x
    for d in range(3):
        lo, hi = [slice(None)] * 3, [slice(None)] * 3
        lo[d], hi[d] = slice(None, -1), slice(1, None)
        y[tuple(lo)] -= x[tuple(hi)]
        y[tuple(hi)] -= x[tuple(lo)]
    return y


def _loop64(c, sino):
    g = _Geometry(c)
    y = sino.double()

    def proj(x):
        return _siddon64(g, x) if c["pair"] == "siddonvi" else _rs64(g, x, False)

    x = torch.zeros((g.nz, g.ny, g.nx), dtype=torch.float64, device=DEVICE)
    res = []
    if c["op"] == "sirt":
        r, b = proj(torch.ones_like(x)), _vi64(g, torch.ones_like(y))
        r = torch.where(r > 0.0, 1.0 / r, torch.zeros_like(r))
        b = torch.where(b > 0.0, 1.0 / b, torch.zeros_like(b))
        for _ in range(c["iters"]):
            e = y - proj(x)
            res.append(float((e * e).sum()))
            x = x + b * _vi64(g, e * r)
        return {"volume": x, "residual": np.array(res)}
    d, gg_prev = None, 0.0
    for k in range(c["iters"]):
        e = y - proj(x)
        res.append(float((e * e).sum()))
        grad = -2.0 * _vi64(g, e) + 2.0 * LAMBDA * _laplacian64(_laplacian64(x))
        gg = float((grad * grad).sum())
        d = grad if c["op"] == "gd" or k == 0 else gg / gg_prev * d + grad
        gg_prev = gg
        pd, ld = proj(d), _laplacian64(d)
        down = 2.0 * float((pd * pd).sum()) + LAMBDA * 2.0 * float((ld * ld).sum())
        x = x - float((grad * d).sum()) / down * d
    return {"volume": x, "residual": np.array(res)}


def exact(case, seed):
    c = case
    if c["op"] == "serve":
        return [_loop64(p, _sinogram(_Geometry(p), seed + 101 * i))["volume"] for i, p in enumerate(_parts(c))]
    if c["op"] in LOOPS:
        return _loop64(c, _sinogram(_Geometry(c), seed))
    if _Geometry(c).updates > EXACT_MOST:
        return None
    g, x, scale, out_scale = _data(c, seed)
    x = x.double() / scale
    if c["op"] == "siddon":
        r = _siddon64(g, x)
    elif c["op"] == "rs":
        r = _rs64(g, x, c["cube"])
    elif c["op"] in ("vi", "fdk"):
        r = _vi64(g, x, c["op"] == "fdk")
    elif c["op"] == "vi_t":
        r = _vi64(g, None, vol=x)
    elif c["op"] == "rs_t":
        r = _rs64(g, None, c["cube"], sino=x)
    else:
        r = _siddon64(g, None, sino=x)
    return r * out_scale
