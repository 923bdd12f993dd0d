"""The work that programs on this library give it, as measurable cases.

Every case goes through a public entry point with the inputs a caller holds:
device arrays for the C ABI's ``*_device`` functions, ``deposit_batch_device``
and ``BatchPlan``, host arrays for ``sphMapping``.  The particle sets are the
distributions of ``sph2grid.workloads`` (uniform box, lattice blast, cluster,
all-sky shell), drawn on the GPU from the seed; the sizes are those of the
benchmark workloads plus small, odd and ragged ones.

``exact`` restates each deposit in 64 bits with plain torch, from the
formulas of the pixel-overlap deposit, the RING-scheme disc deposit, the
triangular-shaped cloud and the nearest-neighbour density.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sphtogrid.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import sph2grid as s2g  # noqa: E402
from sph2grid import _lib  # noqa: E402

KERNELS = {"cubic": s2g.Cubic, "quintic": s2g.Quintic, "wendlandc2": s2g.WendlandC2,
           "wendlandc4": s2g.WendlandC4, "wendlandc6": s2g.WendlandC6,
           "wendlandc8": s2g.WendlandC8}
# flops of one shape(u), by kernel
SHAPE_FLOPS = {"cubic": 6, "quintic": 16, "wendlandc2": 6, "wendlandc4": 9, "wendlandc6": 11,
               "wendlandc8": 14}
DTYPES = {"f32": (torch.float32, _lib.S2G_F32), "f64": (torch.float64, _lib.S2G_F64)}
DEV = "cuda:0"


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: one host-side sphMapping of a thumbnail, as an
        # interactive session or a per-object loop makes thousands of
        dict(name="host_thumbnail", kind="host2d", set="plain", n=4096, npix=64, nq=1,
             kernel="cubic", dtype="f64", calc_mean=False),
        # an ordinary small map on resident particles: latency counts
        dict(name="plain_2d", kind="map2d", set="plain", n=65536, npix=256, nq=1,
             kernel="cubic", dtype="f64", calc_mean=False),
        # a blast on a jittered lattice: all particles of one mid-size hsml,
        # density and temperature in one call, mean values
        dict(name="sedov_2d", kind="map2d", set="sedov", n=1 << 20, npix=1024, nq=2,
             kernel="wendlandc6", dtype="f32", calc_mean=True),
        # a simulation box's cluster, the large production map: hsml from
        # below a pixel to 400 pixels
        dict(name="cluster_2d", kind="map2d", set="cluster", n=1 << 24, npix=4096, nq=1,
             kernel="wendlandc6", dtype="f32", calc_mean=False),
        # a zoomed object: odd sizes, double precision, three quantities
        dict(name="ragged_2d", kind="map2d", set="cluster", n=150001, npix=777, nq=3,
             kernel="quintic", dtype="f64", calc_mean=False),
        # the cluster as a volume
        dict(name="cluster_3d", kind="map3d", set="cluster", n=1 << 24, npix=256, nq=1,
             kernel="wendlandc6", dtype="f32", calc_mean=False),
        # a small volume, odd side, double precision
        dict(name="ragged_3d", kind="map3d", set="plain", n=200003, npix=101, nq=1,
             kernel="cubic", dtype="f64", calc_mean=False),
        # a set of maps of mixed sizes made in one call (every halo of a
        # catalogue)
        dict(name="batch_16", kind="batch", set="sedov", maps=16, n_lo=10000, n_hi=1000000,
             side_lo=128, side_hi=2048, nq=3, kernel="wendlandc6", dtype="f32", calc_mean=True),
        # a serving loop: the same two maps remade from updated inputs
        dict(name="replay_2", kind="plan", set="plain", maps=2, n_lo=30000, n_hi=100000,
             side_lo=200, side_hi=300, nq=1, kernel="cubic", dtype="f64", calc_mean=False),
        # the full sky: density and temperature of one shell of particles
        dict(name="allsky_2maps", kind="allsky", set="shell", n=1 << 22, nside=1024, maps=2,
             kernel="wendlandc4", dtype="f64", calc_mean=True),
        # the same shell on a regular grid
        dict(name="tsc_512", kind="tsc", set="shell", n=1 << 22, npix=512, dtype="f64",
             periodic=False),
        # densities and smoothing lengths of particles that carry none
        dict(name="density_k64", kind="density", set="halos", n=1 << 20, k=64,
             kernel="wendlandc4", dtype="f32", periodic=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host2d", "map2d", "map2d", "map3d", "batch", "plan", "allsky", "tsc",
                       "density"])
    kernel = rng.choice(sorted(KERNELS))
    dtype = rng.choice(["f32", "f64"])
    if kind == "host2d":
        return dict(kind=kind, set=rng.choice(["plain", "sedov"]), n=_log_int(rng, 2000, 40000),
                    npix=_log_int(rng, 32, 300), nq=rng.choice([1, 1, 2]), kernel=kernel,
                    dtype=dtype, calc_mean=rng.random() < 0.5)
    if kind == "map2d":
        return dict(kind=kind, set=rng.choice(["plain", "sedov", "cluster"]),
                    n=_log_int(rng, 4000, 1 << 21), npix=_log_int(rng, 64, 2048),
                    nq=rng.choice([1, 1, 2, 3]), kernel=kernel, dtype=dtype,
                    calc_mean=rng.random() < 0.5)
    if kind == "map3d":
        return dict(kind=kind, set=rng.choice(["plain", "cluster"]),
                    n=_log_int(rng, 4000, 1 << 21), npix=_log_int(rng, 24, 256), nq=1,
                    kernel=kernel, dtype=dtype, calc_mean=False)
    if kind in ("batch", "plan"):
        lo = _log_int(rng, 3000, 30000)
        return dict(kind=kind, set=rng.choice(["plain", "sedov"]), maps=rng.randint(2, 12),
                    n_lo=lo, n_hi=lo * rng.randint(4, 20), side_lo=64,
                    side_hi=rng.choice([300, 512, 1024]), nq=rng.choice([1, 2, 3]),
                    kernel=kernel, dtype=dtype, calc_mean=rng.random() < 0.5)
    if kind == "allsky":
        nside = 2 ** rng.randint(5, 10)
        return dict(kind=kind, set="shell", n=_log_int(rng, 4000, (1 << 21)), nside=nside,
                    maps=rng.randint(1, 3), kernel=kernel, dtype="f64",
                    calc_mean=rng.random() < 0.5)
    if kind == "tsc":
        return dict(kind=kind, set="shell", n=_log_int(rng, 4000, 1 << 22),
                    npix=_log_int(rng, 24, 512), dtype=dtype, periodic=rng.random() < 0.5)
    return dict(kind=kind, set="halos", n=_log_int(rng, 4000, 1 << 20), k=_log_int(rng, 12, 128),
                kernel=kernel, dtype=dtype, periodic=rng.random() < 0.5)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + 7919 * salt + 12345) % (1 << 62))
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float64)


def _sphere(g, n):
    v = _randn(g, n, 3)
    return v / v.norm(dim=1, keepdim=True)


def _particles(which, n, nq, g):
    """x (n x 3, box or shell centred on the origin), h, m, rho, q (n or n x
    nq), w in 64 bits: the sets of sph2grid.workloads."""
    if which == "plain":
        x = _rand(g, n, 3) - 0.5
        m = torch.full((n,), 1.0 / n, device=DEV, dtype=torch.float64)
        h = 2.0 * n ** (-1.0 / 3.0) * torch.exp(0.3 * _randn(g, n))
        rho = 64.0 * m / (4.0 / 3.0 * math.pi * h ** 3)
        q0 = rho.clone()
    elif which == "sedov":
        side = int(math.ceil(n ** (1.0 / 3.0) - 1e-9))
        ids = torch.arange(side ** 3, device=DEV)
        if side ** 3 > n:
            ids = ids[torch.randperm(side ** 3, generator=g, device=DEV)[:n].sort().values]
        c = torch.stack([ids // (side * side), (ids // side) % side, ids % side], 1).double()
        x = (c + 0.5) / side - 0.5 + 0.01 / side * (2.0 * _rand(g, n, 3) - 1.0)
        r = x.norm(dim=1)
        rho = 1.0 + 4.0 * torch.exp(-(r - 0.3) ** 2 / 0.002)
        m = rho / side ** 3
        h = (3.0 * 64.0 * m / (4.0 * math.pi * rho)) ** (1.0 / 3.0)
        q0 = rho.clone()
    elif which == "cluster":
        nh = int(round(0.8 * n))
        halo = _sphere(g, nh) * (1e-3 + (0.5 - 1e-3) * _rand(g, nh, 1))
        x = torch.cat([halo, _rand(g, n - nh, 3) - 0.5])
        h = torch.exp(math.log(1e-4) + math.log(1e3) * _rand(g, n))
        m = torch.full((n,), 1.0 / n, device=DEV, dtype=torch.float64)
        rho = 64.0 * m / (4.0 / 3.0 * math.pi * h ** 3)
        q0 = torch.exp(math.log(1e7) + _randn(g, n))
    else:  # shell, density ~ 1/r
        rad = torch.sqrt(_rand(g, n, 1) * (1.0 - 0.05 ** 2) + 0.05 ** 2)
        x = _sphere(g, n) * rad
        h = torch.exp(math.log(1e-3) + math.log(50.0) * _rand(g, n))
        m = torch.full((n,), 1.0 / n, device=DEV, dtype=torch.float64)
        rho = 64.0 * m / (4.0 / 3.0 * math.pi * h ** 3)
        q0 = rho.clone()
    q = [q0]
    if nq > 1:
        q.append(1e4 * (1.0 + 100.0 * torch.exp(-(x ** 2).sum(1) / 0.01)))
    while len(q) < nq:
        q.append(torch.exp(math.log(1e-6) + 0.8 * _randn(g, n)))
    q = torch.stack(q, 1).contiguous() if nq > 1 else q[0]
    return dict(x=x, h=h, m=m, rho=rho, q=q, w=rho.clone())


def _cast(p, dtype):
    dt = DTYPES[dtype][0]
    return {k: v.to(dt).contiguous() for k, v in p.items()}


def _map_sizes(case):
    """(n, npix) of a batch's maps: spread over the case's ranges, the same
    for every seed (a batch's shape is the program's, its particles are the
    data's)."""
    r = np.random.default_rng(case["maps"] * 7919 + case["n_lo"])
    out = []
    for _ in range(case["maps"]):
        n = int(math.exp(r.uniform(math.log(case["n_lo"]), math.log(case["n_hi"]))))
        s = int(math.exp(r.uniform(math.log(case["side_lo"]), math.log(case["side_hi"]))))
        out.append((n, s))
    return out


def _halos(case, seed):
    """Clustered tracers in the unit box: Plummer-like clumps on a uniform
    background."""
    g, n = _gen(seed), case["n"]
    nb = n // 5
    nc = 64
    cen = _rand(g, nc, 3)
    which = torch.randint(0, nc, (n - nb,), generator=g, device=DEV)
    rad = 0.02 * _rand(g, n - nb, 1) ** 2 + 1e-5
    x = torch.cat([cen[which] + _sphere(g, n - nb) * rad, _rand(g, nb, 3)])
    x = (x - x.floor())[torch.randperm(n, generator=g, device=DEV)]
    x = x.clamp(0.0, 1.0 - 1e-6)
    m = torch.exp(0.2 * _randn(g, n)) / n
    dt = DTYPES[case["dtype"]][0]
    return x.to(dt).contiguous(), m.to(dt).contiguous()


def _sky(case, seed):
    """The shell's particles and each map's quantity and weight: density
    first, then temperatures."""
    g = _gen(seed)
    p = _particles("shell", case["n"], 1, g)
    qs = [p["q"]] + [torch.exp(math.log(1e7) + _randn(g, case["n"]))
                     for _ in range(case["maps"] - 1)]
    return p, qs, [p["w"]] * case["maps"]


def _maps_of(case, seed):
    """The resident particles and outputs of a batch's maps, as
    deposit_batch_device takes them."""
    maps = []
    for k, (n, side) in enumerate(_map_sizes(case)):
        p = _cast(_particles(case["set"], n, case["nq"], _gen(seed, k + 1)), case["dtype"])
        out = torch.empty(case["nq"] * side * side, device=DEV, dtype=torch.float64)
        maps.append(dict(pos=p["x"], hsml=p["h"], m=p["m"], rho=p["rho"], bin_q=p["q"],
                         weights=p["w"], out=out, n=n, nq=case["nq"], npix=side,
                         len2pix=float(side), kernel=KERNELS[case["kernel"]](2),
                         calc_mean=case["calc_mean"], reduce_image=True))
    return maps


def prepare(case, seed):
    kind = case["kind"]
    ctx = s2g.default_context()
    st = {"case": case, "ctx": ctx}
    if kind == "host2d":
        p = _cast(_particles(case["set"], case["n"], case["nq"], _gen(seed)), case["dtype"])
        h = {k: v.cpu().numpy() for k, v in p.items()}
        h["x"] = np.ascontiguousarray(h["x"].T)
        if case["nq"] > 1:
            h["q"] = np.ascontiguousarray(h["q"].T)
        st["p"] = h
        st["par"] = s2g.mappingParameters(x_lim=[-0.5, 0.5], y_lim=[-0.5, 0.5],
                                          z_lim=[-0.5, 0.5], Npixels=case["npix"])
        st["kernel"] = KERNELS[case["kernel"]](2)
    elif kind in ("map2d", "map3d"):
        dims = 2 if kind == "map2d" else 3
        nd = case["npix"] ** dims
        st["p"] = _cast(_particles(case["set"], case["n"], case["nq"], _gen(seed)), case["dtype"])
        st["image"] = torch.empty((case["nq"] + 1) * nd, device=DEV, dtype=torch.float64)
        st["map"] = torch.empty(case["nq"] * nd, device=DEV, dtype=torch.float64)
        st["par"] = _lib.Params(npixels=case["npix"], len2pix=float(case["npix"]))
    elif kind in ("batch", "plan"):
        st["maps"] = _maps_of(case, seed)
        if kind == "plan":
            torch.cuda.synchronize()
            st["plan"] = s2g.BatchPlan(st["maps"], dtype=case["dtype"])
    elif kind == "allsky":
        st["p"], st["qs"], st["ws"] = _sky(case, seed)
        np_ = 12 * case["nside"] ** 2
        st["out"] = [torch.empty(np_, device=DEV, dtype=torch.float64)
                     for _ in range(2 * case["maps"])]
    elif kind == "tsc":
        p = _cast(_particles("shell", case["n"], 1, _gen(seed)), case["dtype"])
        st["p"] = {"x": p["x"], "q": p["q"]}
        st["par"] = _lib.Params(npixels=case["npix"], len2pix=case["npix"] / 2.0)
        st["grid"] = torch.empty(2 * case["npix"] ** 3, device=DEV, dtype=torch.float64)
    else:
        st["x"], st["m"] = _halos(case, seed)
        st["rho"] = torch.empty(case["n"], device=DEV, dtype=torch.float64)
        st["hsml"] = torch.empty(case["n"], device=DEV, dtype=torch.float64)
        st["box"] = (C.c_double * 3)(1.0, 1.0, 1.0) if case["periodic"] else None
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _vp(t):
    return C.c_void_p(t.data_ptr())


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def run(st):
    case, ctx = st["case"], st["ctx"]
    lib, kind = ctx.lib, case["kind"]
    if kind == "host2d":
        p = st["p"]
        # sphMapping centres Pos in place, so a caller who maps it again
        # passes a copy
        return s2g.sphMapping(p["x"].copy(), p["h"], p["m"], p["rho"], p["q"], p["w"],
                              param=st["par"], kernel=st["kernel"], show_progress=False,
                              calc_mean=case["calc_mean"])
    if kind in ("map2d", "map3d"):
        dims = 2 if kind == "map2d" else 3
        p = st["p"]
        ctx.check(lib.s2g_deposit_device(
            ctx.handle, dims, DTYPES[case["dtype"]][1], _vp(p["x"]), _vp(p["h"]), _vp(p["m"]),
            _vp(p["rho"]), _vp(p["q"]), case["nq"], _vp(p["w"]), case["n"], C.byref(st["par"]),
            KERNELS[case["kernel"]].kernel_id, dims,
            _lib.S2G_FLAG_CALC_MEAN if case["calc_mean"] else 0, _vp(st["image"]), _stream(),
            None), "deposit")
        ctx.check(lib.s2g_reduce_device(ctx.handle, dims, case["npix"], case["nq"],
                                        _lib.S2G_FLAG_REDUCE, _vp(st["image"]), _vp(st["map"]),
                                        _stream()), "reduce")
        return {"image": st["image"], "map": st["map"]}
    if kind == "batch":
        s2g.deposit_batch_device(st["maps"], dtype=case["dtype"],
                                 stream=torch.cuda.current_stream().cuda_stream)
        return [m["out"] for m in st["maps"]]
    if kind == "plan":
        st["plan"].run(stream=torch.cuda.current_stream().cuda_stream)
        return [m["out"] for m in st["maps"]]
    if kind == "allsky":
        p, nm = st["p"], case["maps"]
        ptrs = lambda ts: (C.c_void_p * len(ts))(*[t.data_ptr() for t in ts])  # noqa: E731
        ctx.check(lib.s2g_healpix_deposit_maps_device(
            ctx.handle, _lib.S2G_F64, _vp(p["x"]), _vp(p["h"]), _vp(p["m"]), _vp(p["rho"]), nm,
            ptrs(st["qs"]), ptrs(st["ws"]), case["n"], case["nside"],
            KERNELS[case["kernel"]].kernel_id, 2,
            _lib.S2G_FLAG_CALC_MEAN if case["calc_mean"] else 0, ptrs(st["out"][:nm]),
            ptrs(st["out"][nm:]), _stream(), None), "allsky")
        return st["out"]
    if kind == "tsc":
        p = st["p"]
        ctx.check(lib.s2g_tsc3d_device(
            ctx.handle, DTYPES[case["dtype"]][1], _vp(p["x"]), _vp(p["q"]), case["n"],
            C.byref(st["par"]), _lib.S2G_FLAG_PERIODIC if case["periodic"] else 0,
            _vp(st["grid"]), _stream()), "tsc")
        return st["grid"]
    ctx.check(lib.s2g_mass_density_device(
        ctx.handle, DTYPES[case["dtype"]][1], _vp(st["x"]), _vp(st["m"]), case["n"],
        KERNELS[case["kernel"]].kernel_id, 3, case["k"], st["box"], _vp(st["rho"]),
        _vp(st["hsml"]), _stream(), None), "density")
    return {"rho": st["rho"], "hsml": st["hsml"]}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _mean_h(which, n, power):
    """Mean of hsml^power (box or shell lengths) over a set's distribution."""
    if which == "plain":
        return (2.0 * n ** (-1.0 / 3.0)) ** power * math.exp(0.5 * (0.3 * power) ** 2)
    if which == "sedov":
        side = math.ceil(n ** (1.0 / 3.0) - 1e-9)
        return (48.0 / (math.pi * side ** 3)) ** (power / 3.0)
    a, b = (1e-4, 1e-1) if which == "cluster" else (1e-3, 5e-2)
    return (b ** power - a ** power) / (power * math.log(b / a))


def _map_work(which, n, npix, nq, dims, kernel, dtype):
    """Inputs read and planes written once; per pixel inside a particle's
    kernel disc (ball) its distance, shape and one multiply-add per plane."""
    size = 4 if dtype == "f32" else 8
    nd = npix ** dims
    vol = math.pi if dims == 2 else 4.0 / 3.0 * math.pi
    # a disc as wide as the image is counted once per pixel
    pix = n * max(1.0, min(vol * _mean_h(which, n, dims), 1.0) * nd)
    return (n * (6 + nq) * size + nd * (2 * nq + 1) * 8,
            pix * (5 + dims + SHAPE_FLOPS[kernel] + 2 * (nq + 1)))


def work(case):
    kind = case["kind"]
    if kind in ("host2d", "map2d", "map3d"):
        b, f = _map_work(case["set"], case["n"], case["npix"], case["nq"],
                         3 if kind == "map3d" else 2, case["kernel"], case["dtype"])
    elif kind in ("batch", "plan"):
        b = f = 0.0
        for n, side in _map_sizes(case):
            bb, ff = _map_work(case["set"], n, side, case["nq"], 2, case["kernel"],
                               case["dtype"])
            b, f = b + bb, f + ff
    elif kind == "allsky":
        npx = 12 * case["nside"] ** 2
        # disc of angle h / r: mean h^2 times mean 1 / r^2 of the shell
        inv_r2 = 2.0 * math.log(1.0 / 0.05) / (1.0 - 0.05 ** 2)
        pix = case["n"] * max(1.0, _mean_h("shell", 1, 2) * inv_r2 / 4.0 * npx)
        b = case["n"] * (6 + 2 * case["maps"]) * 8 + 2 * case["maps"] * npx * 8
        f = pix * (20 + SHAPE_FLOPS[case["kernel"]] + 4 * case["maps"])
    elif kind == "tsc":
        size = 4 if case["dtype"] == "f32" else 8
        b = case["n"] * 4 * size + 2 * case["npix"] ** 3 * 8
        f = case["n"] * (27 * 5 + 40)
    else:
        size = 4 if case["dtype"] == "f32" else 8
        b = case["n"] * (4 * size + 16)
        f = case["n"] * (case["k"] + 1) * (9 + SHAPE_FLOPS[case["kernel"]])
    return {"bytes": float(b), "flops": float(f)}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
_CHUNK = 1 << 25      # expanded (particle, pixel) pairs at a time
_MOST = 3_000_000_000  # pairs beyond which a restatement takes too long


def _shape(kernel, u):
    t = (1.0 - u).clamp(min=0.0)
    if kernel == "cubic":
        return torch.where(u < 0.5, 1.0 + 6.0 * (u - 1.0) * u * u, 2.0 * t ** 3)
    if kernel == "quintic":
        a, b = (2.0 / 3.0 - u).clamp(min=0.0), (1.0 / 3.0 - u).clamp(min=0.0)
        return t ** 5 - 6.0 * a ** 5 + 15.0 * b ** 5
    if kernel == "wendlandc2":
        return t ** 4 * (1.0 + 4.0 * u)
    if kernel == "wendlandc4":
        return t ** 6 * (1.0 + u * (6.0 + u * (35.0 / 3.0)))
    if kernel == "wendlandc6":
        return t ** 8 * (1.0 + u * (8.0 + u * (25.0 + u * 32.0)))
    return t ** 10 * (1.0 + u * (10.0 + u * (42.0 + u * (90.0 + u * (429.0 / 5.0)))))


def _norm3(kernel):
    return {"cubic": 8.0, "quintic": 2187.0 / 40.0, "wendlandc2": 10.5,
            "wendlandc4": 495.0 / 32.0, "wendlandc6": 1365.0 / 64.0,
            "wendlandc8": 1785.0 / 64.0}[kernel] / math.pi


def _expand(counts):
    """(owner, rank within owner) of counts[i] entries per i."""
    own = torch.repeat_interleave(torch.arange(counts.numel(), device=DEV), counts)
    first = torch.cumsum(counts, 0) - counts
    return own, torch.arange(own.numel(), device=DEV) - first[own]


def _slices(counts):
    """Consecutive index ranges whose counts add up to about _CHUNK."""
    c = torch.cumsum(counts, 0).cpu().numpy()
    a = 0
    while a < c.size:
        base = c[a - 1] if a else 0
        b = int(np.searchsorted(c, base + _CHUNK, side="right"))
        b = max(b, a + 1)
        yield a, b
        a = b


def _sums(v, counts):
    """Sums of counts[i] consecutive values of v per i."""
    return torch.segment_reduce(v, "sum", lengths=counts, unsafe=True)


def _deposit64(p, npix, len2pix, nq, kernel, calc_mean, dims):
    """Flat image, (nq + 1) planes of npix^dims, or None if it takes too long."""
    p = {k: v.double() for k, v in p.items()}
    q = p["q"].reshape(-1, nq)
    h = p["h"] * len2pix
    xs = p["x"][:, :dims] * len2pix + 0.5 * npix
    lo = torch.floor(xs - h[:, None]).clamp(min=0)
    hi = torch.floor(xs + h[:, None]).clamp(max=npix - 1)
    wid = (hi - lo + 1).clamp(min=0).long()
    cnt = wid.prod(1)
    if not calc_mean:
        cnt = torch.where((q != 0).any(1), cnt, torch.zeros_like(cnt))
    if int(cnt.sum()) > _MOST:
        return None
    if dims == 2:
        # (2h)^2 * w * m / rho' / (2h)^2 with rho' = rho / len2pix^3
        num = p["w"] * p["m"] / p["rho"] * len2pix ** 3
    else:
        num = p["w"] * p["m"] / p["rho"] * len2pix ** 4
    nd = npix ** dims
    img = torch.zeros(nq + 1, nd, device=DEV, dtype=torch.float64)
    for a, b in _slices(cnt):
        own, r = _expand(cnt[a:b])
        own = own + a
        hh = h[own]
        idx = torch.zeros_like(r)
        s2 = torch.zeros_like(hh)
        ov = torch.ones_like(hh)
        for d in range(dims - 1, -1, -1):
            wd = wid[own, d]
            c = lo[own, d] + (r % wd)
            r = r // wd
            x = xs[own, d]
            ov = ov * (torch.minimum(x + hh, c + 1.0) - torch.maximum(x - hh, c))
            s2 = s2 + (x - c - 0.5) ** 2
            idx = idx + c.long() * npix ** (dims - 1 - d)
        u = torch.sqrt(s2) / hh
        wk = _shape(kernel, u) * ov
        tot, area = _sums(wk, cnt[a:b]), _sums(ov, cnt[a:b])
        fb = tot == 0
        wk = torch.where(fb[own - a], ov, wk)
        den = torch.where(fb, area, tot)
        pw = wk * torch.where(den != 0, num[a:b] / den, torch.zeros_like(den))[own - a]
        img[nq].index_add_(0, idx, pw)
        for k in range(nq):
            img[k].index_add_(0, idx, pw * q[own, k])
    return img


def _reduced2d(img, npix, nq):
    w = img[nq]
    out = [torch.where(w > 0, img[k] / w, img[k]).view(npix, npix).t().reshape(-1)
           for k in range(nq)]
    return torch.cat(out)


def _allsky64(p, qs, ws, nside, kernel, calc_mean):
    """Maps then weight maps, or None if it takes too long."""
    x, h = p["x"], p["h"]
    dx = x.norm(dim=1)
    ok = dx >= h
    x, h, dx = x[ok], h[ok], dx[ok]
    mrho = (p["m"] / p["rho"])[ok]
    npix = 12 * nside * nside
    th = torch.asin(h / dx)
    if float((th * th).sum()) / 4.0 * npix > _MOST / 2:
        return None
    ang = math.sqrt(4.0 * math.pi / npix)
    theta = torch.atan2(torch.hypot(x[:, 0], x[:, 1]), x[:, 2])
    phi = torch.atan2(x[:, 1], x[:, 0])
    phi = torch.where(phi < 0, phi + 2 * math.pi, phi)
    # rings 1 .. 4 nside - 1: colatitude, pixels, first pixel, half-pixel shift
    r = torch.arange(1, 4 * nside, device=DEV)
    rn = torch.minimum(r, 4 * nside - r)
    cap = rn < nside
    zc = torch.where(cap, 1.0 - rn.double() ** 2 / (3.0 * nside * nside),
                     (2 * nside - rn).double() * 2.0 / (3.0 * nside))
    # south of the equator the colatitude cosine changes sign
    z = torch.where(cap, torch.where(r > 2 * nside, -zc, zc),
                    (2 * nside - r).double() * 2.0 / (3.0 * nside))
    nr = torch.where(cap, 4 * rn, torch.full_like(r, 4 * nside))
    start = torch.cumsum(nr, 0) - nr
    shift = torch.where(cap, 0.5, torch.where(((r - nside) % 2) == 0, 0.5, 0.0)).double()
    tr = torch.acos(z)
    # the ring range of each disc: rings whose colatitude lies within th
    lo = torch.searchsorted(tr, (theta - th).contiguous())
    hi = torch.searchsorted(tr, (theta + th).contiguous(), right=True)
    nring = (hi - lo).clamp(min=0)
    part, k = _expand(nring)
    ring = lo[part] + k
    # azimuth half-width of the disc on the ring (haversine form)
    st, sr = torch.sin(theta)[part], torch.sin(tr)[ring]
    hav = torch.sin(0.5 * th[part]) ** 2 - torch.sin(0.5 * (tr[ring] - theta[part])) ** 2
    f = hav / (st * sr)
    dphi = torch.where(f >= 1.0, torch.full_like(f, math.pi),
                       2.0 * torch.asin(torch.sqrt(f.clamp(0.0, 1.0))))
    full = (f >= 1.0) & (hav > 0)
    nrr = nr[ring].double() / (2 * math.pi)
    ilo = torch.floor(nrr * (phi[part] - dphi) - shift[ring]) + 1
    ihi = torch.floor(nrr * (phi[part] + dphi) - shift[ring])
    cnt = torch.where(hav > 0, (ihi - ilo + 1).clamp(min=0), torch.zeros_like(ilo)).long()
    cnt = torch.where(full, nr[ring], torch.minimum(cnt, nr[ring]))
    del st, sr, hav, f, dphi, full, nrr, ihi

    # the pixel that holds the particle
    zz = torch.cos(theta)
    za = zz.abs()
    tt = (phi / (0.5 * math.pi)) % 4.0
    jp = torch.floor(nside * (0.5 + tt - 0.75 * zz)).long()
    jm = torch.floor(nside * (0.5 + tt + 0.75 * zz)).long()
    ir = nside + 1 + jp - jm
    ks = 1 - (ir & 1)
    ip = torch.remainder((jp + jm - nside + ks + 1) // 2, 4 * nside)
    eq = 2 * nside * (nside - 1) + (ir - 1) * 4 * nside + ip
    tmp = nside * torch.sqrt(3.0 * (1.0 - za))
    tp = tt - torch.floor(tt)
    ir2 = torch.floor(tp * tmp).long() + torch.floor((1.0 - tp) * tmp).long() + 1
    ip2 = torch.remainder(torch.floor(tt * ir2).long(), 4 * ir2)
    pol = torch.where(zz > 0, 2 * ir2 * (ir2 - 1) + ip2, npix - 2 * ir2 * (ir2 + 1) + ip2)
    cpix = torch.where(za <= 2.0 / 3.0, eq, pol)

    def terms(pp, pix_theta, pix_phi):
        """distance, kernel weight and area weight of pixels of particles pp"""
        a = torch.sin(0.5 * (pix_theta - theta[pp])) ** 2 + torch.sin(pix_theta) * \
            torch.sin(theta[pp]) * torch.sin(0.5 * (pix_phi - phi[pp])) ** 2
        d = 2.0 * torch.asin(torch.sqrt(a.clamp(0.0, 1.0)))
        ar = (th[pp] - (d - 0.5 * ang)).abs().clamp(max=ang) / ang
        u = d / th[pp]
        return torch.where(u < 1.0, _shape(kernel, u), torch.zeros_like(u)) * ar, ar

    def ring_of(pix):
        return torch.searchsorted(start, pix.contiguous(), right=True) - 1

    np_ = x.shape[0]
    tot = torch.zeros(np_, device=DEV, dtype=torch.float64)
    area = torch.zeros(np_, device=DEV, dtype=torch.float64)
    has = torch.zeros(np_, device=DEV, dtype=torch.bool)

    def chunks():
        for a, b in _slices(cnt):
            e, k = _expand(cnt[a:b])
            e = e + a
            pp, rg = part[e], ring[e]
            m = ilo[e].long() + k
            pix = start[rg] + torch.remainder(m, nr[rg])
            yield pp, pix, tr[rg], (m.double() + shift[rg]) * 2 * math.pi / nr[rg]

    for pp, pix, pt, ph in chunks():
        w, ar = terms(pp, pt, ph)
        tot.index_add_(0, pp, w)
        area.index_add_(0, pp, ar)
        has[pp[pix == cpix[pp]]] = True
    miss = torch.nonzero(~has).reshape(-1)
    cr = ring_of(cpix[miss])
    cphi = ((cpix[miss] - start[cr]).double() + shift[cr]) * 2 * math.pi / nr[cr]
    wm, am = terms(miss, tr[cr], cphi)
    tot.index_add_(0, miss, wm)
    area.index_add_(0, miss, am)
    fb = tot == 0
    den = torch.where(fb, area, tot)
    base = torch.where(den != 0, mrho / (ang * dx) ** 2 / den, torch.zeros_like(den))
    maps = [torch.zeros(npix, device=DEV, dtype=torch.float64) for _ in range(2 * len(qs))]

    def add(pp, pix, w, ar):
        pw0 = torch.where(fb[pp], ar, w) * base[pp]
        for i, (q, wt) in enumerate(zip(qs, ws)):
            pw = pw0 * wt[ok][pp]
            if not calc_mean:
                pw = torch.where(q[ok][pp] != 0, pw, torch.zeros_like(pw))
            maps[i].index_add_(0, pix, pw * q[ok][pp])
            maps[len(qs) + i].index_add_(0, pix, pw)

    for pp, pix, pt, ph in chunks():
        add(pp, pix, *terms(pp, pt, ph))
    add(miss, cpix[miss], wm, am)
    return maps


def _tsc64(x, q, npix, len2pix, periodic):
    g = x.double() * len2pix + 0.5 * npix
    q = q.double()
    c = torch.floor(g)
    w = []
    for o in (-1, 0, 1):
        d = (g - (c + o + 0.5)).abs()
        w.append(torch.where(d < 0.5, 0.75 - d * d, 0.5 * (1.5 - d).clamp(min=0.0) ** 2))
    out = torch.zeros(2, npix ** 3, device=DEV, dtype=torch.float64)
    for a in range(3):
        for b in range(3):
            for e in range(3):
                i = c.long() + torch.tensor([a - 1, b - 1, e - 1], device=DEV)
                ww = w[a][:, 0] * w[b][:, 1] * w[e][:, 2]
                if periodic:
                    i = torch.remainder(i, npix)
                else:
                    inside = ((i >= 0) & (i < npix)).all(1)
                    i, ww = i.clamp(0, npix - 1), torch.where(inside, ww, torch.zeros_like(ww))
                k = (i[:, 0] * npix + i[:, 1]) * npix + i[:, 2]
                out[0].index_add_(0, k, q * ww)
                out[1].index_add_(0, k, ww)
    return out.reshape(-1)


def _density64(x, m, k, kernel, periodic):
    x, m = x.double(), m.double()
    n = x.shape[0]
    if n > 150000:
        return None
    rho = torch.empty(n, device=DEV, dtype=torch.float64)
    hs = torch.empty_like(rho)
    rows = max(1, (1 << 27) // n)
    for a in range(0, n, rows):
        d2 = torch.zeros(min(rows, n - a), n, device=DEV, dtype=torch.float64)
        for c in range(3):
            d = (x[a:a + rows, c, None] - x[None, :, c]).abs()
            if periodic:
                d = torch.minimum(d, 1.0 - d)
            d2 += d * d
        v, i = torch.topk(d2, k + 1, dim=1, largest=False)
        r = torch.sqrt(v)
        h = r.max(1).values
        wk = _shape(kernel, r / h[:, None])
        rho[a:a + rows] = (m[i] * wk).sum(1) * _norm3(kernel) / h ** 3
        hs[a:a + rows] = h
    bias = {"wendlandc2": (0.0294, 0.977), "wendlandc4": (0.01342, 1.579),
            "wendlandc6": (0.0116, 2.236)}.get(kernel)
    if bias:
        corr = bias[0] * (k * 0.01) ** -bias[1] * m * _norm3(kernel) / hs ** 3
        rho = torch.where(rho - corr > 0, rho - corr, rho)
    return {"rho": rho, "hsml": hs}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("host2d", "map2d", "map3d"):
        dims = 3 if kind == "map3d" else 2
        npix, nq = case["npix"], case["nq"]
        if _map_work(case["set"], case["n"], npix, nq, dims, case["kernel"], case["dtype"])[1] \
                > 100.0 * _MOST:
            return None
        p = _cast(_particles(case["set"], case["n"], nq, _gen(seed)), case["dtype"])
        if kind == "host2d":
            # sphMapping keeps the centres inside the box
            keep = (p["x"].abs() <= 0.5).all(1)
            p = {k: v[keep] for k, v in p.items()}
        img = _deposit64(p, npix, float(npix), nq, case["kernel"], case["calc_mean"], dims)
        if img is None:
            return None
        if kind == "map3d":
            v = img[0]
            return {"image": img.reshape(-1), "map": torch.where(v > 0, v / img[1], v)}
        red = _reduced2d(img, npix, nq)
        if kind == "host2d":
            return red.cpu().numpy().reshape((npix, npix, nq), order="F")
        return {"image": img.reshape(-1), "map": red}
    if kind in ("batch", "plan"):
        out = []
        for m in _maps_of(case, seed):
            p = dict(x=m["pos"], h=m["hsml"], m=m["m"], rho=m["rho"], q=m["bin_q"],
                     w=m["weights"])
            img = _deposit64(p, m["npix"], m["len2pix"], m["nq"], case["kernel"],
                             case["calc_mean"], 2)
            out.append(None if img is None else _reduced2d(img, m["npix"], m["nq"]))
        return out
    if kind == "allsky":
        return _allsky64(*_sky(case, seed), case["nside"], case["kernel"], case["calc_mean"])
    if kind == "tsc":
        p = _cast(_particles("shell", case["n"], 1, _gen(seed)), case["dtype"])
        return _tsc64(p["x"], p["q"], case["npix"], case["npix"] / 2.0, case["periodic"])
    x, m = _halos(case, seed)
    return _density64(x, m, case["k"], case["kernel"], case["periodic"])
