"""The projections a user runs, as measurable cases.

``listed()`` names the cases, ``draw(rng)`` gives another one of the same
ranges, ``prepare`` makes what a program holds before the call (the cloud, its
rays on the host or on the GPU, the fields being fitted), ``run`` is one call
through the public API, ``work`` the bytes and FP64 operations it cannot do
without, and ``exact`` the same outputs by brute force over all generators in
plain FP64 torch (small cases only).

Meshes are made on the GPU from the seed alone: ``uniform`` points, or
``clustered`` ones -- 70 % of the points in 200 clumps of power-law sizes with
r^-2 profiles, the rest a uniform background, no two points closer than about
1e-5 of the box -- which is the kind of mesh the projection is used on.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import vortrace_amd as vt
from vortrace_amd import synthetic

DEV = "cuda"


# ------------------------------------------------------------------ cases ----

def _case(kind, mesh, n, nx, ny, *, periodic, mode="sum", nf=1, box=100.0, views=1,
          rotate=False, name=None):
    c = dict(kind=kind, mesh=mesh, n=n, nx=nx, ny=ny, periodic=periodic, mode=mode, nf=nf,
             box=box, views=views, rotate=rotate)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # One sight line, traced cell by cell (the smallest call: latency).
        _case("trace1", "uniform", 20_000, 1, 1, periodic=False, name="one_ray"),
        # A thumbnail of a small periodic box.
        _case("grid", "uniform", 5_000, 16, 16, periodic=True, box=10.0, name="thumb_16"),
        # An ordinary map of a uniform 100k box, numpy in and out.
        _case("grid", "uniform", 100_000, 128, 128, periodic=False, name="uniform_128"),
        # Three fields at once, odd image sides, an oblique camera, points
        # outside the box filtered by the padding rule.
        _case("grid", "clustered", 300_000, 257, 301, periodic=False, nf=3, rotate=True,
              name="fields_oblique"),
        # Sight lines in random directions with their segments (catalogues).
        _case("trace", "clustered", 200_000, 19_997, 1, periodic=False, name="traced_20k"),
        # The peak density along each pixel of a deep map.
        _case("grid", "clustered", 700_000, 384, 384, periodic=True, mode="max",
              name="max_384"),
        # The column map of a 2M cosmological box, rays and image on the GPU.
        _case("tensor", "clustered", 2_000_000, 512, 512, periodic=True, name="column_512"),
        # A volume rendering at screen size.
        _case("grid", "clustered", 1_000_000, 1024, 1024, periodic=True, mode="volume", nf=4,
              name="volume_1024"),
        # One step of fitting the densities to a column map.
        _case("fit", "clustered", 2_000_000, 512, 512, periodic=True, name="fit_512"),
        # One step of fitting colours and opacities to a rendering.
        _case("fit", "clustered", 1_000_000, 256, 256, periodic=True, mode="volume", nf=4,
              name="volume_fit_256"),
        # A fly-through: cameras of many directions, extents and sizes at once.
        _case("views", "clustered", 4_000_000, 512, 512, periodic=True, views=12, rotate=True,
              name="cameras_4m"),
        # The largest: a fit step of an 8M mesh against four maps.
        _case("fit", "clustered", 8_000_000, 512, 512, periodic=True, views=4, rotate=True,
              name="fit_8m"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trace1", "grid", "grid", "tensor", "trace", "fit", "views"])
    periodic = rng.random() < 0.6
    mesh = rng.choice(["uniform", "clustered", "clustered"])
    n = _log_int(rng, 5_000, 2_000_000)
    nx = _log_int(rng, 16, 512)
    ny = max(16, min(600, int(nx * rng.uniform(0.6, 1.4))))
    mode, nf = rng.choice([("sum", 1), ("sum", 1), ("sum", 3), ("volume", 4), ("max", 1),
                           ("min", 2)])
    if kind == "trace1":
        return _case(kind, mesh, _log_int(rng, 5_000, 200_000), 1, 1, periodic=False)
    if kind == "trace":
        return _case(kind, mesh, _log_int(rng, 5_000, 400_000), _log_int(rng, 100, 30_000), 1,
                     periodic=False)
    if kind == "fit":
        if mode in ("max", "min"):
            mode, nf = "sum", 1
        return _case(kind, mesh, n, nx, ny, periodic=periodic, mode=mode, nf=nf)
    if kind == "views":
        return _case(kind, mesh, n, 256, 256, periodic=periodic, views=rng.randint(2, 6),
                     rotate=True)
    return _case(kind, mesh, n, nx, ny, periodic=periodic, mode=mode, nf=nf,
                 rotate=periodic is False and rng.random() < 0.5)


# ----------------------------------------------------------------- meshes ----

def _separate(pos, box):
    """Keeps one point per cell of a fine grid, moved into the cell's middle
    half: no two points are closer than half a cell (1e-5 of the box)."""
    h = box * 2e-5
    k = torch.clamp((pos / h).floor().to(torch.int64), 0, int(round(box / h)) - 1)
    side = int(round(box / h))
    key = (k[:, 0] * side + k[:, 1]) * side + k[:, 2]
    order = torch.argsort(key, stable=True)
    s = key[order]
    first = torch.ones_like(s, dtype=torch.bool)
    first[1:] = s[1:] != s[:-1]
    keep = torch.sort(order[first])[0]
    frac = pos[keep] / h - k[keep].to(pos.dtype)
    return (k[keep].to(pos.dtype) + 0.25 + 0.5 * frac.clamp(0, 1)) * h, keep


def _symmetry(case, seed):
    """The seed's symmetry of the box: an order of the axes and which are
    reflected.  Sight lines are traced through one mesh per size, turned by it
    and with its points in another order and other densities: the segments of
    all rays then are as many for every seed, as a caller with buffers has it."""
    rng = np.random.default_rng(seed + 3)
    return rng.permutation(3), rng.integers(0, 2, 3).astype(np.float64)


def _turn(x, case, seed):
    order, flip = _symmetry(case, seed)
    if isinstance(x, torch.Tensor):
        order = torch.from_numpy(order.copy()).to(x.device)
        flip = torch.from_numpy(flip).to(x.device)
    x = x[:, order]
    return flip * (case["box"] - x) + (1.0 - flip) * x


def _traced(case):
    return case["kind"] in ("trace", "trace1")


def _mesh(case, seed):
    """(pos (n, 3), rho (n,)) on the GPU, FP64."""
    if not _traced(case):
        return _points(case, seed)
    pos, rho = _points(case, 1)
    g = torch.Generator(device=DEV)
    g.manual_seed(seed + 19)
    order = torch.argsort(torch.rand(len(pos), generator=g, device=DEV))
    rho = rho * torch.exp(0.1 * torch.randn(len(pos), generator=g, device=DEV,
                                            dtype=torch.float64))
    return _turn(pos, case, seed)[order].contiguous(), rho[order]


def _chords(case, seed):
    """Start and end points of sight lines in random directions."""
    rng = np.random.default_rng(11)
    ab = case["box"] * (0.02 + 0.96 * rng.random((2, case["nx"], 3)))
    return [np.ascontiguousarray(_turn(x, case, seed)) for x in ab]


def _points(case, seed):
    n, box = case["n"], case["box"]
    g = torch.Generator(device=DEV)
    g.manual_seed(1_000_003 * (seed % 2_000_000_011) + 17)

    def u(*shape):
        return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64)

    def z(*shape):
        return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float64)

    if case["mesh"] == "uniform":
        return u(n, 3) * box, torch.exp(z(n))
    m = int(n * 1.1)
    ncl = int(0.7 * m)
    centres = u(200, 3) * box
    w = 1.0 / (1.0 - u(200))
    w = torch.minimum(w, w.sum() / 20.0)
    which = torch.searchsorted(torch.cumsum(w / w.sum(), 0), u(ncl)).clamp(max=199)
    rs = 5e-4 * box * (100.0 ** u(200))
    rad = rs[which] * (0.01 + 0.99 * u(ncl))
    v = z(ncl, 3)
    v = v / v.norm(dim=1, keepdim=True)
    pos = torch.cat([centres[which] + rad[:, None] * v, u(m - ncl, 3) * box])
    frac = (w / w.sum())[which] * 0.7
    dens = torch.cat([frac * n / (4.0 * math.pi * rad * rad * rs[which]),
                      torch.full((m - ncl,), 0.3 * n / box ** 3, device=DEV,
                                 dtype=torch.float64)])
    perm = torch.argsort(u(m))
    pos, dens = torch.remainder(pos[perm], box), dens[perm]
    pos, keep = _separate(pos, box)
    dens = dens[keep]
    if len(pos) < n:  # saturated clumps: fill up with background points
        extra, _ = _separate(u(2 * (n - len(pos)) + 64, 3) * box, box)
        extra = extra[: n - len(pos)] + box * 1e-6
        pos = torch.cat([pos, extra])
        dens = torch.cat([dens, torch.full((len(extra),), 0.3 * n / box ** 3, device=DEV,
                                           dtype=torch.float64)])
    pos, dens = pos[:n], dens[:n]
    return pos, dens * torch.exp(0.3 * z(len(pos)))


def _fields(case, rho):
    """Field columns on the host: rho, rho and two derived fields, or RGBA."""
    r = rho.cpu().numpy()
    if case["nf"] == 1:
        return r
    if case["nf"] == 4:
        return synthetic.rgba_transfer(r, 0.7 * case["box"] ** 2 / len(r))
    return np.column_stack([r, np.sqrt(r), r * r])[:, : case["nf"]].copy()


def _views(case, seed):
    """grid_projection arguments of the case's cameras."""
    box, ext = case["box"], case["box"]
    rng = np.random.default_rng(seed + 5)
    c = [box / 2] * 3
    out = []
    for i in range(case["views"]):
        nres = (case["nx"], case["ny"])
        if case["kind"] == "views":
            nres = min((64, 128, 256, 512, 1024)[i % 5], 2 * case["nx"])
            ext = box * (0.1 + 0.9 * rng.random())
        lo, hi = box / 2 - ext / 2, box / 2 + ext / 2
        v = dict(extent=[lo, hi], nres=nres, bounds=[0.0, box], center=c)
        if case["rotate"]:
            v.update(yaw=float(2 * np.pi * rng.random()),
                     pitch=float(np.arccos(2 * rng.random() - 1)), roll=0.0)
        out.append(v)
    return out


# ------------------------------------------------------------ prepare, run ----

def prepare(case, seed):
    pos, rho = _mesh(case, seed)
    box = case["box"]
    f = _fields(case, rho)
    bb = [0.0, box] * 3
    kw = {}
    if not case["periodic"]:
        kw["vol"] = np.full(len(pos), box ** 3 / len(pos))
    pc = vt.ProjectionCloud(pos.cpu().numpy(), f, boundbox=bb, periodic=case["periodic"], **kw)
    st = dict(case=case, pc=pc)
    kind = case["kind"]
    if _traced(case):
        st["start"], st["end"] = _chords(case, seed)
        if kind == "trace1":
            st["start"], st["end"] = st["start"][0], st["end"][0]
    else:
        st["views"] = _views(case, seed)
    if kind in ("tensor", "fit"):
        s, e = [], []
        for v in st["views"]:
            a, b = vt.grid.generate_projection_grid(**v)
            s.append(torch.from_numpy(a.reshape(-1, 3)))
            e.append(torch.from_numpy(b.reshape(-1, 3)))
        st["start"], st["end"] = torch.cat(s).to(DEV), torch.cat(e).to(DEV)
        pc.set_ray_rows(case["ny"])
    if kind == "fit":
        g = torch.Generator(device=DEV)
        g.manual_seed(seed + 7)
        fd = torch.from_numpy(f).to(DEV)
        st["fields"] = fd.requires_grad_(True)
        nout = 3 if case["mode"] == "volume" else case["nf"]
        rays = st["start"].shape[0]
        st["weight"] = torch.randn((rays, nout) if nout > 1 else (rays,), generator=g,
                                   device=DEV, dtype=torch.float64)
    return st


def run(st):
    case, pc = st["case"], st["pc"]
    kind, mode = case["kind"], case["mode"]
    if kind == "trace1":
        return pc.traced_projection(st["start"], st["end"], reduction=mode)
    if kind == "trace":
        return pc.traced_projection(st["start"], st["end"], reduction=mode, flatten=True)
    if kind == "grid":
        return pc.grid_projection(**st["views"][0], reduction=mode)
    if kind == "tensor":
        return pc.projection_tensor(st["start"], st["end"], reduction=mode)
    if kind == "views":
        return pc.batch_grid_projection(st["views"], reduction=mode)
    # one fit step: the image and the gradient of a loss linear in it
    fields = st["fields"]
    fields.grad = None
    img = pc.projection_grad(st["start"], st["end"], fields, reduction=mode)
    (img * st["weight"]).sum().backward()
    return img.detach(), fields.grad


# -------------------------------------------------------------- work, exact ----

def _nrays(case):
    if case["kind"] == "views":
        return sum(min((64, 128, 256, 512, 1024)[i % 5], 2 * case["nx"]) ** 2
                   for i in range(case["views"]))
    return case["views"] * case["nx"] * case["ny"]


def work(case):
    """Each ray's end points in and its values out, every cell's generator and
    fields in once, and per crossing (about 1.1 n^(1/3) a ray, half that for
    chords) one bisector of two generators: about 30 FP64 operations for each
    of the some 16 neighbours a cell has.  A fit step adds the image's
    gradient in, the fields' gradient out and a multiply-add per crossing and
    field; a traced projection writes 24 bytes per crossing."""
    rays = _nrays(case)
    nout = 3 if case["mode"] == "volume" else case["nf"]
    cross = rays * 1.1 * case["n"] ** (1.0 / 3.0)
    if _traced(case):
        cross *= 0.5
    nbytes = rays * (48 + 8 * nout) + case["n"] * (24 + 8 * case["nf"])
    flops = cross * (16 * 30 + 4 * nout)
    if case["kind"] == "fit":
        nbytes += rays * 8 * nout + case["n"] * 8 * case["nf"]
        flops += cross * 4 * case["nf"]
    if _traced(case):
        nbytes += cross * 24
    return {"bytes": float(nbytes), "flops": float(flops)}


def _brute_trace(gen, ids, a, b):
    """Cells and boundaries of rays a -> b by the lower envelope of all
    generators' distances along each ray.  Lists of per-step (cell (R,),
    s_enter (R,), s_exit (R,)); finished rays repeat with zero length."""
    d = b - a
    length = d.norm(dim=1)
    d = d / length[:, None]
    rows = torch.arange(len(a), device=a.device)
    rel2 = ((gen * gen).sum(1)[None, :] - 2.0 * (a @ gen.T))
    proj = d @ gen.T
    c = torch.argmin(rel2, dim=1)
    s = torch.zeros_like(length)
    steps = []
    while True:
        den = 2.0 * (proj - proj[rows, c][:, None])
        cross = (rel2 - rel2[rows, c][:, None]) / den
        cross = torch.where(den > 1e-12, cross, math.inf)
        cross[rows, c] = math.inf
        nxt = torch.argmin(cross, dim=1)
        ex = torch.minimum(torch.maximum(cross[rows, nxt], s), length)
        steps.append((ids[c], s, ex))
        c = torch.where(ex < length, nxt, c)
        s = ex
        if bool((s >= length).all()):
            return steps


def exact(case, seed):
    kind, mode = case["kind"], case["mode"]
    images = 27 if case["periodic"] else 1
    if case["rotate"] or kind == "views" or case["n"] * images * _nrays(case) > 2.5e9:
        return None
    pos, rho = _mesh(case, seed)
    f = torch.from_numpy(np.asarray(_fields(case, rho))).to(DEV).reshape(case["n"], -1)
    box = case["box"]
    ids = torch.arange(case["n"], device=DEV)
    gen, gid = pos, ids
    if case["periodic"]:
        sh = torch.cartesian_prod(*[torch.arange(-1, 2, device=DEV, dtype=torch.float64)] * 3)
        gen = (pos[None] + box * sh[:, None]).reshape(-1, 3)
        gid = ids.repeat(27)
    if _traced(case):
        a, b = [torch.from_numpy(x).to(DEV) for x in _chords(case, seed)]
    else:
        x = (torch.arange(case["nx"], device=DEV, dtype=torch.float64) + 0.5) * box / case["nx"]
        y = (torch.arange(case["ny"], device=DEV, dtype=torch.float64) + 0.5) * box / case["ny"]
        xy = torch.cartesian_prod(x, y)
        a = torch.cat([xy, torch.zeros_like(xy[:, :1])], 1)
        b = torch.cat([xy, torch.full_like(xy[:, :1], box)], 1)
    nout = 3 if mode == "volume" else case["nf"]
    out = torch.empty((len(a), nout), dtype=torch.float64, device=DEV)
    grad = torch.zeros_like(f)
    segs = []
    chunk = max(1, int(5e7 // len(gen)))
    if kind == "fit":
        g = torch.Generator(device=DEV)
        g.manual_seed(seed + 7)
        weight = torch.randn((len(a), nout) if nout > 1 else (len(a),), generator=g, device=DEV,
                             dtype=torch.float64).reshape(len(a), nout)
    for i in range(0, len(a), chunk):
        steps = _brute_trace(gen, gid, a[i:i + chunk], b[i:i + chunk])
        cell = torch.stack([q[0] for q in steps], 1)
        s0 = torch.stack([q[1] for q in steps], 1)
        s1 = torch.stack([q[2] for q in steps], 1)
        ds = s1 - s0
        live = ds > 0
        leaf = f.clone().requires_grad_(kind == "fit")
        val = leaf[cell]
        if mode == "sum":
            img = (val * ds[..., None]).sum(1)
        elif mode == "max":
            img = torch.where(live[..., None], val, -math.inf).amax(1)
        elif mode == "min":
            img = torch.where(live[..., None], val, math.inf).amin(1)
        else:
            tr = torch.exp(-val[..., 3] * ds)
            before = torch.cumprod(torch.cat([torch.ones_like(tr[:, :1]), tr[:, :-1]], 1), 1)
            img = ((before * (1.0 - tr))[..., None] * val[..., :3]).sum(1)
        if kind == "fit":
            (img * weight[i:i + chunk]).sum().backward()
            grad += leaf.grad
        out[i:i + chunk] = img.detach()
        if _traced(case):
            segs.append(((0.5 * (s0 + s1))[live], ds[live]))
    img = out[:, 0] if nout == 1 else out
    if kind == "fit":
        return img, grad.reshape(-1) if case["nf"] == 1 else grad
    if kind == "tensor":
        return out
    if _traced(case):
        mid = torch.cat([q[0] for q in segs]).cpu().numpy()
        ds = torch.cat([q[1] for q in segs]).cpu().numpy()
        if kind == "trace1":
            return np.float64(out[0, 0].item()), None, mid, ds
        return img.cpu().numpy(), None, mid, ds, None
    shape = (case["nx"], case["ny"]) + ((nout,) if nout > 1 else ())
    return img.reshape(shape).cpu().numpy()
