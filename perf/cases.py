"""The work that users of this framework have it do, as timed cases.

A case is one pass through the public entry points (fluidtissue_amd's Python
API, and the C ABI where that is how a device-resident program calls it) on
inputs that stay on the device as in a simulation loop: a level set arrives in
phi, the pass turns it into the distance field (or advects it), and the
outputs are what a simulation goes on with.

Kinds:
  reinit    LevelSet::resetPhi_ with its blend, phi resident in HBM; distance
            to the crossing points (the reference's own) or to the triangles,
            full domain or a narrow band
  points    EuclideanDistance::init / resetPhi, the drop-in on host arrays
  batch     many independent fields in one captured graph (parameter sweeps)
  normals   the reinit with level-set normals, then the surface tension, which
            takes the interface curvature (the growth program's step)
  advect    the advection step of LevelSet::update on device arrays
  update    LevelSet::update on host arrays: advection, then the reinit with
            the update blend (the leveque program's step)

Sizes: grids of 16 to 256 nodes per axis, the range of the reference's own
parameter files and of bench.py; non-cubic and odd ones among them.  Meshes
are the Kuhn grids of the library's generator, with and without the jitter
that stands for an unstructured mesh.
"""
import ctypes as C
import math

import numpy as np
import torch

import fluidtissue_amd as fa
from fluidtissue_amd import _lib

DEV = "cuda:0"


def listed():
    def c(name, kind, nx, ny, nz, **kw):
        d = dict(name=name, kind=kind, nx=nx, ny=ny, nz=nz, jitter=0.0, field="spheres", mode="triangles",
                 blend="init", band_h=0.0)
        d.update(kw)
        return d
    return [
        # the smallest call: a coarse trial run, bound by launches and latency
        c("points_32", "reinit", 32, 32, 32, field="sphere_wave", mode="points"),
        # a non-cubic domain with the update blend, odd sizes
        c("triangles_47x33x17_update", "reinit", 47, 33, 17, field="ellipsoids", blend="update"),
        # the drop-in class in an unchanged host program
        c("dropin_points_61", "points", 61, 61, 61, field="ellipsoids", mode="points"),
        # a narrow band around one smooth surface
        c("band6h_star_128", "reinit", 128, 128, 128, field="star", band_h=6.0),
        # the everyday 3-D run: unstructured mesh, update blend, many surfaces
        c("triangles_127_update", "reinit", 127, 127, 127, jitter=0.2, blend="update"),
        # the largest reinit, to the triangles and to the reference's points
        c("triangles_256", "reinit", 256, 256, 256, jitter=0.2),
        c("points_256", "reinit", 256, 256, 256, jitter=0.2, mode="points", blend="update"),
        # a narrow band at the largest size
        c("band6h_256", "reinit", 256, 256, 256, jitter=0.2, band_h=6.0),
        # a sweep of small runs as one captured graph
        c("batch_64", "batch", 24, 96, 64, field="ellipsoids"),
        # growth's step: distance, normals, curvature and surface tension
        c("normals_160x144x131", "normals", 160, 144, 131, jitter=0.2),
        # the advection of a device-resident run
        c("advect_200", "advect", 200, 200, 200, jitter=0.2),
        # leveque's step from a host program
        c("update_host_72", "update", 72, 72, 72, jitter=0.1, field="sphere_wave", mode="points", blend="update"),
    ]


def draw(rng):
    kind = rng.choice(["reinit"] * 6 + ["points", "batch", "normals", "normals", "advect", "advect", "update"])
    top = {"reinit": 248, "points": 72, "normals": 150, "advect": 180, "update": 84, "batch": 96}[kind]
    n = int(round(math.exp(rng.uniform(math.log(16 if kind != "batch" else 24), math.log(top)))))
    d = dict(kind=kind, nx=n, ny=n, nz=n, jitter=rng.choice([0.0, 0.1, 0.2]),
             field=rng.choice(["spheres", "spheres", "ellipsoids", "star", "sphere_wave"]),
             mode=rng.choice(["triangles", "triangles", "points"]), blend=rng.choice(["init", "update"]), band_h=0.0)
    if kind == "batch":                         # nx..ny: range of the fields' sizes; nz: fields
        d.update(nx=rng.randint(16, 24), ny=max(26, n), nz=rng.randint(5, 56), jitter=0.0, field="ellipsoids")
        return d
    if rng.random() < 0.5:                      # non-cubic
        d.update(ny=max(9, int(n * rng.uniform(0.5, 1.0))), nz=max(9, int(n * rng.uniform(0.4, 1.0))))
    if kind == "reinit" and rng.random() < 0.35:
        d["band_h"] = round(rng.uniform(2.0, 9.0), 2)
    if kind in ("points", "update"):
        d["mode"] = "points"
    if kind == "update":
        d["blend"] = "update"
    return d


# ---- inputs -------------------------------------------------------------------
def _h(case):
    return 1.0 / (max(case["nx"], case["ny"], case["nz"]) - 1)


def _grid(nx, ny, nz, h):
    """Node coordinates of an unjittered grid, x-major, as floats."""
    ax = [(torch.arange(n, dtype=torch.float64, device=DEV) * h).to(torch.float32) for n in (nx, ny, nz)]
    return torch.stack(torch.meshgrid(*ax, indexing="ij"), -1).reshape(-1, 3)


def _field(kind, xyz, seed):
    """Level set (float64) of the benchmark's kinds, its shape drawn from the seed."""
    g = np.random.default_rng(1000 + seed)
    x = xyz.to(torch.float64)
    if kind == "sphere_wave":                   # sign right, slope far from 1
        p = torch.from_numpy(0.35 + 0.04 * g.uniform(-1, 1, 3)).to(DEV)
        wave = 1.0 + 0.5 * torch.sin(4 * math.pi * x).prod(1)
        return (torch.linalg.vector_norm(x - p, dim=1) - (0.15 + 0.01 * g.uniform())) * wave
    if kind == "star":                          # r = 0.3 + 0.06 cos 5 phi sin^3 theta
        p = torch.from_numpy(0.5 + 0.02 * g.uniform(-1, 1, 3)).to(DEV)
        q = x - p
        r = torch.linalg.vector_norm(q, dim=1).clamp_min(1e-12)
        st = torch.sqrt((1 - (q[:, 2] / r) ** 2).clamp_min(0))
        return (r - (0.3 + 0.06 * torch.cos(5 * torch.atan2(q[:, 1], q[:, 0]) + g.uniform()) * st ** 3)) * 2.3
    ext = x.max(0).values.cpu().numpy()
    phi = torch.full((x.shape[0],), math.inf, dtype=torch.float64, device=DEV)
    if kind == "spheres":                       # 64 spheres over the domain
        for c, r in zip(g.uniform(0.1, 0.9, (64, 3)), g.uniform(0.02, 0.08, 64)):
            torch.minimum(phi, torch.linalg.vector_norm(x - torch.from_numpy(c * ext).to(DEV), dim=1) - r, out=phi)
        return 1.5 * phi
    for _ in range(int(g.integers(1, 17))):     # a union of ellipsoids
        c, a = g.uniform(0.25, 0.75, 3) * ext, g.uniform(0.03, 0.2, 3)
        q, _ = np.linalg.qr(g.standard_normal((3, 3)))
        y = (x - torch.from_numpy(c).to(DEV)) @ torch.from_numpy(q).to(DEV) / torch.from_numpy(a).to(DEV)
        torch.minimum(phi, (torch.linalg.vector_norm(y, dim=1) - 1.0) * float(a.min()), out=phi)
    return phi


def _flow(xyz):
    """Rotation about the vertical axis plus a shear, |V| <= 0.9; then the pressure."""
    x = xyz.to(torch.float64)
    v = [-(x[:, 1] - 0.5), x[:, 0] - 0.5, 0.2 * torch.sin(2 * math.pi * x[:, 0])]
    return torch.cat(v + [torch.zeros_like(x[:, 0])])


def _resident(case, seed):
    """A handle with the case's mesh made on the device, and the node coordinates."""
    r = fa.Reinit(0)
    dims = (case["nx"], case["ny"], case["nz"])
    r.set_kuhn_batch([dims], jitter=case["jitter"], seed=seed, spacings=[_h(case)])
    if case["jitter"] == 0.0:
        return r, _grid(*dims, _h(case))
    xyz = np.empty((r.n, 3), np.float32)
    _lib.check(_lib.lib.ft_get_mesh(r._h, xyz.ctypes.data_as(C.c_void_p), None, None, None))
    return r, torch.from_numpy(xyz).to(DEV)


def prepare(case, seed):
    kind = case["kind"]
    h = _h(case)
    if kind == "batch":
        sizes = [int(n) for n in np.random.default_rng(7).integers(case["nx"], case["ny"] + 1, case["nz"])]
        r = fa.Reinit(0)
        r.set_kuhn_batch(sizes)
        phi0 = torch.cat([_field(case["field"], _grid(n, n, n, 1.0 / (n - 1)), 100 * seed + k)
                          for k, n in enumerate(sizes)])
        return dict(case=case, r=r, phi0=phi0, phi=torch.empty_like(phi0))
    if kind == "points":
        m = fa.kuhn_mesh((case["nx"], case["ny"], case["nz"]), spacing=h)
        phi = _field(case["field"], torch.from_numpy(m.xyz).to(DEV), seed).cpu().numpy()
        p = phi[m.edges]
        e = m.edges[(p[:, 0] < 0) != (p[:, 1] < 0)]
        t = (phi[e[:, 0]] / (phi[e[:, 0]] - phi[e[:, 1]]))[:, None]
        ifp = ((1 - t) * m.xyz[e[:, 0]].astype(np.float64) + t * m.xyz[e[:, 1]]).astype(np.float32)
        d = fa.EuclideanDistance(0)
        d.init(m.xyz)
        return dict(case=case, d=d, ifp=ifp, phi0=phi)
    if kind == "update":
        m = fa.kuhn_mesh((case["nx"], case["ny"], case["nz"]), spacing=h, jitter=case["jitter"], seed=seed)
        r = fa.Reinit(0)
        r.set_mesh(m)
        x = torch.from_numpy(m.xyz).to(DEV)
        return dict(case=case, r=r, phi0=_field(case["field"], x, seed).cpu().numpy(), flow=_flow(x).cpu().numpy(),
                    dt=0.5 * h / 0.9)
    r, xyz = _resident(case, seed)
    phi0 = _field(case["field"], xyz, seed)
    s = dict(case=case, r=r, phi0=phi0, phi=torch.empty_like(phi0))
    if kind == "advect":
        s.update(flow=_flow(xyz), dt=0.5 * h / 0.9, info=_lib.FtAdvectInfo())
    else:
        s["ifn"] = torch.empty_like(phi0)
    if kind == "normals":
        s["force"] = [torch.empty_like(phi0) for _ in range(3)]
    return s


# ---- one pass -----------------------------------------------------------------
def _counts(c):
    return [int(c.n_ifp), int(c.n_tri), int(c.n_if_elems), int(c.n_clamped)]


def run(s):
    case = s["case"]
    kind = case["kind"]
    kw = dict(mode=case["mode"], blend=case["blend"], band=case["band_h"] * _h(case))
    if kind == "points":
        phi = s["phi0"].copy()
        s["d"].reset_phi(s["ifp"], len(s["ifp"]), phi)
        return dict(phi=phi)
    if kind == "update":
        phi, ifn, cnt, info = s["r"].update(s["phi0"], s["flow"], s["dt"], tol=1e-10, mode="points")
        return dict(phi=phi, ifn=ifn)
    stream = torch.cuda.current_stream().cuda_stream
    s["phi"].copy_(s["phi0"])                   # the level set of this step
    if kind == "advect":
        _lib.check(_lib.lib.ft_advect_device(s["r"]._h, C.c_void_p(s["phi"].data_ptr()),
                                             C.c_void_p(s["flow"].data_ptr()), s["dt"], 1e-10, 1000,
                                             C.byref(s["info"]), C.c_void_p(stream)))
        return dict(phi=s["phi"])
    if kind == "batch":
        per = s["r"].reset_phi_graph_device(s["phi"].data_ptr(), None, stream=stream, **kw)
        return dict(phi=s["phi"], counts=np.array([_counts(c) for c in per]))
    if kind == "normals":
        r, f = s["r"], s["force"]
        cnt = r.reset_phi_device(s["phi"].data_ptr(), s["ifn"].data_ptr(), stream=stream, want_normals=True, **kw)
        for a in f:
            a.zero_()
        _lib.check(_lib.lib.ft_surface_tension_device(r._h, C.c_float(0.1), C.c_int32(1), *[C.c_void_p(a.data_ptr()) for a in f],
                                                      C.c_void_p(stream)))
        return dict(phi=s["phi"], ifn=s["ifn"], fx=f[0], fy=f[1], fz=f[2], counts=np.array(_counts(cnt)))
    cnt = s["r"].reset_phi_device(s["phi"].data_ptr(), s["ifn"].data_ptr(), stream=stream, **kw)
    return dict(phi=s["phi"], ifn=s["ifn"], counts=np.array(_counts(cnt)))


# ---- what one pass cannot do without -------------------------------------------
def work(case):
    """Bytes: coordinates and phi of each node read, phi (and phi_ifn) written,
    each tet's node ids read; the surface terms are left out (they grow with
    the square of the size).  Operations: one point-primitive distance per
    node, and per matrix entry or tet where the path has them."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["kind"] == "batch":
        sizes = np.random.default_rng(7).integers(nx, ny + 1, nz)
        n, t = int((sizes ** 3).sum()), int((6 * (sizes - 1) ** 3).sum())
    else:
        n, t = nx * ny * nz, 6 * (nx - 1) * (ny - 1) * (nz - 1)
    reinit = dict(bytes=28 * n + 8 * n + 16 * t, flops=60 * n)
    kind = case["kind"]
    if kind == "points":
        return dict(bytes=28 * n, flops=10 * n)
    if kind in ("reinit", "batch"):
        return reinit
    if kind == "normals":
        # tets again for the gradients of phi and of the unit normal; normals and forces per node
        return dict(bytes=reinit["bytes"] + 2 * 16 * t + 60 * n, flops=reinit["flops"] + 300 * t)
    # advection: tets, velocity, phi; the matrix (15 entries a row: value and
    # column) once per product, two products and the vectors per iteration,
    # about 10 iterations
    adv = dict(bytes=16 * t + 56 * n + 10 * (2 * 15 * 12 + 100) * n, flops=10 * 2 * 30 * n + 600 * t)
    if kind == "update":
        return dict(bytes=adv["bytes"] + reinit["bytes"], flops=adv["flops"] + reinit["flops"])
    return adv


# ---- the same in 64 bits -------------------------------------------------------
PERM = ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0))
EDGES = ((0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3))


def _tets(nx, ny, nz):
    """Kuhn tets of the grid: six per cell, each a monotone path 000 -> 111."""
    i, j, k = torch.meshgrid(torch.arange(nx - 1), torch.arange(ny - 1), torch.arange(nz - 1), indexing="ij")
    base = ((i * ny + j) * nz + k).reshape(-1)
    step = (ny * nz, nz, 1)
    out = []
    for p in PERM:
        v = [base]
        for a in p:
            v.append(v[-1] + step[a])
        out.append(torch.stack(v, 1))
    return torch.stack(out, 1).reshape(-1, 4).to(DEV)


def _cross(x, phi, a, b):
    t = (phi[a] / (phi[a] - phi[b]))[:, None]
    return (1 - t) * x[a] + t * x[b]


def _triangles(x, phi, tets):
    """Marching tets: one triangle for one node cut off, two for two and two."""
    neg = phi[tets] < 0
    nn = neg.sum(1)
    tris = []
    for sel in ((nn == 1) | (nn == 3), nn == 2):
        t, s = tets[sel], neg[sel]
        cut = torch.stack([s[:, a] != s[:, b] for a, b in EDGES], 1)
        if not len(t):
            continue
        m = int(cut[0].sum())
        which = cut.nonzero()[:, 1].reshape(-1, m)                     # the cut edges in local order
        ea = torch.tensor([e[0] for e in EDGES], device=DEV)[which]
        eb = torch.tensor([e[1] for e in EDGES], device=DEV)[which]
        p = [_cross(x, phi, t.gather(1, ea[:, q:q + 1])[:, 0], t.gather(1, eb[:, q:q + 1])[:, 0]) for q in range(m)]
        for q in ((0, 1, 2),) if m == 3 else ((0, 2, 3), (0, 1, 3)):
            tris.append(torch.stack([p[q[0]], p[q[1]], p[q[2]]], 1))
    return torch.cat(tris)


def _triangle_distance(x, tri):
    """Nearest distance of each point to the triangles, by brute force in chunks."""
    a, b, c = tri[:, 0], tri[:, 1], tri[:, 2]
    nrm = torch.linalg.cross(b - a, c - a)
    nn = (nrm * nrm).sum(1)
    out = torch.empty(len(x), dtype=torch.float64, device=DEV)
    step = max(1, 20_000_000 // max(1, len(tri)))
    for i in range(0, len(x), step):
        q = x[i:i + step, None, :]
        best, inside = None, nn[None, :] > 0
        for u, v in ((a, b), (b, c), (c, a)):
            e = v - u
            w = q - u
            t = ((w * e).sum(-1) / (e * e).sum(-1).clamp_min(1e-300)).clamp(0, 1)
            d2 = ((w - t[..., None] * e) ** 2).sum(-1)
            best = d2 if best is None else torch.minimum(best, d2)
            inside = inside & ((torch.linalg.cross(e.expand_as(w), w) * nrm).sum(-1) >= 0)
        plane = ((q - a) * nrm).sum(-1) ** 2 / nn.clamp_min(1e-300)
        out[i:i + step] = torch.sqrt(torch.where(inside, plane, best).min(1).values)
    return out


def _point_distance(x, p):
    out = torch.empty(len(x), dtype=torch.float64, device=DEV)
    step = max(1, 60_000_000 // max(1, len(p)))
    for i in range(0, len(x), step):
        d2 = sum((x[i:i + step, c:c + 1] - p[None, :, c]) ** 2 for c in range(3))
        out[i:i + step] = torch.sqrt(d2.min(1).values)
    return out


def _advected(x, tets, phi, flow, dt):
    """Crank-Nicolson on the P1 Galerkin form, (M + s A) y = (M - s A) phi, to round-off."""
    n = len(x)
    p = x[tets]                                                        # (T, 4, 3)
    B = (p[:, 1:] - p[:, :1]).transpose(1, 2)
    det = torch.linalg.det(B).abs()
    g = torch.linalg.inv(B)                                            # rows: gradients of basis 1..3
    G = torch.cat([-g.sum(1, keepdim=True), g], 1)                     # (T, 4, 3)
    al, be = (5 + 3 * math.sqrt(5)) / 20, (5 - math.sqrt(5)) / 20      # degree-2 rule: exact for both forms
    sh = torch.full((4, 4), be, dtype=torch.float64, device=DEV)
    sh.fill_diagonal_(al)
    V = flow[:3 * n].reshape(3, n).t()[tets]                           # (T, 4, 3)
    Vq = torch.einsum("qj,tjc->tqc", sh, V)
    w = det / 24.0
    Me = torch.einsum("qi,qj->ij", sh, sh)[None] * w[:, None, None]
    Ae = torch.einsum("qi,tqc,tjc->tij", sh, Vq, G) * w[:, None, None]
    i = tets[:, :, None].expand(-1, 4, 4).reshape(-1)
    j = tets[:, None, :].expand(-1, 4, 4).reshape(-1)

    def mat(e):
        return torch.sparse_coo_tensor(torch.stack([i, j]), e.reshape(-1), (n, n)).coalesce().to_sparse_csr()
    L, R = mat(Me + 0.5 * dt * Ae), mat(Me - 0.5 * dt * Ae)
    b = R @ phi
    diag = torch.zeros(n, dtype=torch.float64, device=DEV)
    diag.index_add_(0, tets.reshape(-1), torch.diagonal(Me + 0.5 * dt * Ae, dim1=1, dim2=2).reshape(-1))
    y, r = phi.clone(), b - L @ phi                                    # BiCGSTAB, Jacobi
    r0, rho, alpha, om = r.clone(), 1.0, 1.0, 1.0
    v = q = torch.zeros_like(r)
    for _ in range(200):
        if float(r.norm()) <= 1e-15 * float(b.norm()):
            break
        rho1 = float(r0 @ r)
        q = r + (rho1 / rho) * (alpha / om) * (q - om * v)
        yh = q / diag
        v = L @ yh
        alpha = rho1 / float(r0 @ v)
        sres = r - alpha * v
        z = sres / diag
        t = L @ z
        om = float(t @ sres) / max(float(t @ t), 1e-300)
        y, r, rho = y + alpha * yh + om * z, sres - om * t, rho1
    return y


def exact(case, seed):
    kind, dims = case["kind"], (case["nx"], case["ny"], case["nz"])
    n = dims[0] * dims[1] * dims[2]
    if kind in ("batch", "normals", "update") or case["jitter"] != 0.0:
        return None
    x32 = _grid(*dims, _h(case))
    x, phi = x32.to(torch.float64), _field(case["field"], x32, seed)
    if kind == "advect":
        if n > 100 ** 3:
            return None
        return dict(phi=_advected(x, _tets(*dims), phi, _flow(x32), 0.5 * _h(case) / 0.9))
    if n > (70 ** 3 if case["mode"] == "points" else 40 ** 3):
        return None
    tets = _tets(*dims)
    cut = torch.unique(torch.cat([tets[:, list(e)] for e in EDGES]), dim=0)
    cut = cut[(phi[cut[:, 0]] < 0) != (phi[cut[:, 1]] < 0)]
    if not len(cut):
        return None
    if case["mode"] == "points":
        d = _point_distance(x, _cross(x, phi, cut[:, 0], cut[:, 1]))
    else:
        d = _triangle_distance(x, _triangles(x, phi, tets))
    if case["band_h"] > 0:
        d = d.clamp_max(case["band_h"] * _h(case))
    ifn = torch.where(phi < 0, -d, d)
    if kind == "points":
        return dict(phi=ifn)
    if case["blend"] == "init":
        return dict(phi=ifn, ifn=ifn, counts=None)
    kept = ifn.clone()
    on = cut.reshape(-1)
    kept[on] = phi[on]                                                 # nodes of the cut edges keep their value
    return dict(phi=0.75 * kept + 0.25 * ifn, ifn=ifn, counts=None)
