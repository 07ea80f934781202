"""The work this package is timed on, through its public entry points.

Every case is one call (or one analysis cycle) of a program that uses
``letkf_amd``: the per-point drop-in on host arrays, batched solves on device
tensors, Lorenz-96 cycles, global (SPEEDY- and GFS-sized) cycles, regional
radar cycles and a batch of served jobs.  Inputs are synthetic, drawn on the
GPU from the seed: smooth ensemble fields, obs of a truth drawn from the same
distribution, obs errors and localisation scales of the configurations in
``letkf_amd.synth``.
"""
import ctypes
import math

import numpy as np
import torch

from letkf_amd import _lib
from letkf_amd.core import letkf_core, letkf_core_batch, make_job
from letkf_amd.das import GlobalLetkf, L96Letkf, RegionalLetkf, run_batch

RE = 6371.3e3
CUT2 = 13.33333333               # squared normalised cutoff distance of the regional grid
SPREAD = 2.0 * math.sqrt(10.0 / 3.0)   # cutoff of the global and Lorenz-96 grids, in scales
ID_U, ID_V, ID_T, ID_Q, ID_PS = 2819, 2820, 3073, 3330, 14593


# --- the cases ---------------------------------------------------------------
def listed():
    return [
        # one grid point of a host program that calls letkf_core itself: latency
        dict(name="core_point_k20", kind="core", k=20, p=60),
        # a batch of points with every optional output (T, w-bar, Pa kept for diagnosis)
        dict(name="batch_trans_k40", kind="batch", npt=4000, k=40, p=250, nobs=20000, prec="f64",
             out="trans", nv=0),
        # device-side pipeline with its own lists, between the eigensolver classes
        dict(name="batch_apply_k80_f32", kind="batch", npt=3001, k=80, p=333, nobs=20011,
             prec="f32", out="apply", nv=5),
        # the smallest served model: N = 40, new obs every cycle
        dict(name="l96_n40_k20", kind="l96", nx=40, k=20),
        # more members than local obs: the p x p solve
        dict(name="l96_n960_k200", kind="l96", nx=960, k=200),
        # the reference's T30 cycle: new obs through the device operator, then the analysis
        dict(name="speedy_k20_cycle", kind="global", nlon=96, nlat=48, nlev=7, k=20, nstation=415,
             obs_lev=7, cap=0, prec="f64", sigma=500.0e3, hx=True, graph=False),
        # the same grid, obs resident, replayed as a graph in the mixed form
        dict(name="speedy_k20_bf16x3", kind="global", nlon=96, nlat=48, nlev=7, k=20,
             nstation=415, obs_lev=7, cap=0, prec="bf16x3", sigma=500.0e3, hx=False, graph=True),
        # large ensemble on a T15-like grid
        dict(name="global_k256", kind="global", nlon=48, nlat=24, nlev=7, k=256, nstation=415,
             obs_lev=7, cap=0, prec="f64", sigma=500.0e3, hx=False, graph=False),
        # GFS-sized grid, lists capped at the 1000 nearest
        dict(name="gfs_k40", kind="global", nlon=192, nlat=94, nlev=64, k=40, nstation=600,
             obs_lev=16, cap=1000, prec="f64", sigma=700.0e3, hx=False, graph=False),
        # a radar subdomain in the split-BF16x3 form
        dict(name="radar_40_bf16x3", kind="regional", nx=40, ny=40, nlev=30, k=50, cap=1000,
             prec="bf16x3", sigma=2000.0, relax=0.0),
        # the radar configuration on a quarter of its columns, plain FP64
        dict(name="radar_128_f64", kind="regional", nx=128, ny=128, nlev=60, k=50, cap=1000,
             prec="f64", sigma=2000.0, relax=0.0),
        # small jobs of several models in shared launches, as the server enqueues them
        dict(name="served_batch", kind="served", nx=240, k1=20, k2=64, k3=120, nlon=48, nlat=24,
             nlev=7, kg=20, nstation=200),
    ]


def draw(rng):
    def logi(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(["core", "batch", "batch", "l96", "global", "global", "regional",
                       "regional"])
    if kind == "core":
        return dict(kind="core", k=logi(4, 128), p=logi(1, 2000))
    if kind == "batch":
        k = logi(5, 94)
        return dict(kind="batch", npt=logi(64, 4001), k=k, p=logi(5, 700), nobs=logi(3000, 30000),
                    prec=rng.choice(["f64", "f32", "bf16x3"]), out=rng.choice(["trans", "apply"]),
                    nv=rng.randint(1, 8))
    if kind == "l96":
        return dict(kind="l96", nx=logi(40, 960), k=logi(10, 200))
    if kind == "global":
        k = logi(10, 200)
        nlon, nlat = (logi(24, 48), logi(12, 24)) if k > 95 else (logi(24, 128), logi(12, 64))
        # the mixed forms on grids whose exact analysis is quick
        nlev = logi(1, 7) if k > 95 else logi(2, 30)
        prec = rng.choice(["f64", "f32", "bf16x3"]) if nlon * nlat * nlev < 40000 else "f64"
        obs_lev = rng.randint(1, min(nlev, 7))
        return dict(kind="global", nlon=nlon, nlat=nlat, nlev=nlev, k=k, nstation=logi(50, 500),
                    obs_lev=obs_lev, cap=rng.choice([0, 0, logi(30, 1000)]), prec=prec,
                    sigma=rng.uniform(300.0e3, 800.0e3), hx=prec == "f64" and rng.random() < 0.5,
                    graph=rng.random() < 0.3)
    return dict(kind="regional", nx=logi(12, 96), ny=logi(12, 96), nlev=logi(4, 60),
                k=logi(12, 90), cap=rng.choice([1000, logi(40, 1000)]), prec="f64",
                sigma=rng.uniform(900.0, 2200.0), relax=rng.choice([0.0, 0.0, 0.7]))


# --- inputs ------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _rand(g, *shape, lo=0.0, hi=1.0):
    return lo + (hi - lo) * torch.rand(shape, generator=g, device="cuda", dtype=torch.float64)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float64)


def _waves(g, n, nz, ny, nx, kmax, modes=12):
    """n random smooth fields (n, nz, ny, nx) of unit variance."""
    z, y, x = (torch.arange(s, device="cuda", dtype=torch.float64) / s for s in (nz, ny, nx))
    pz, py, px = (_rand(g, n, modes, 1, hi=2 * math.pi) for _ in range(3))
    kx = torch.randint(0, kmax, (n, modes, 1), generator=g, device="cuda")
    ky, kz = _rand(g, n, modes, 1, lo=0.3, hi=kmax), _rand(g, n, modes, 1, lo=0.1, hi=2.0)
    fx = torch.cos(2 * math.pi * kx * x + px)
    fy = torch.cos(math.pi * ky * y + py) * _randn(g, n, modes, 1) * math.sqrt(8.0 / modes)
    fz = torch.cos(math.pi * kz * z + pz)
    fyz = (fz[:, :, :, None] * fy[:, :, None, :]).reshape(n, modes, nz * ny)
    return torch.bmm(fyz.transpose(1, 2).contiguous(), fx).reshape(n, nz, ny, nx)


def _host(t):
    """Device tensor whose last index runs fastest -> Fortran-ordered host array of the
    reversed shape."""
    return t.contiguous().cpu().numpy().T


def _global_problem(c, seed):
    """Fields (4 variables + ps), stations and H(x) of every member, in device tensors."""
    g = _gen(seed)
    nlon, nlat, nlev, k = c["nlon"], c["nlat"], c["nlev"], c["k"]
    lon = 360.0 / nlon * np.arange(nlon)
    x, _ = np.polynomial.legendre.leggauss(nlat)
    lat = np.rad2deg(np.arcsin(x))
    sig = (np.array([0.95, 0.835, 0.685, 0.51, 0.34, 0.2, 0.08]) if nlev == 7 else
           np.exp(np.linspace(math.log(0.995), math.log(0.01 if nlev > 30 else 0.08), nlev)))
    sig_t = torch.tensor(sig, device="cuda")
    amp = (10.0, 10.0, 5.0, 5.0e-4, 1000.0)
    base = (0.0 * sig_t, 0.0 * sig_t, 250.0 + 40.0 * sig_t, 8.0e-3 * sig_t ** 3)
    x3 = torch.empty((4, k + 1, nlev, nlat, nlon), device="cuda", dtype=torch.float64)
    for v in range(4):
        mean = base[v][:, None, None] + amp[v] * _waves(g, 1, nlev, nlat, nlon, 9)[0]
        x3[v] = mean + 0.3 * amp[v] * _waves(g, k + 1, nlev, nlat, nlon, 9)
    ps = 1.0e5 + amp[4] * (_waves(g, 1, 1, nlat, nlon, 9) +
                           0.3 * _waves(g, k + 1, 1, nlat, nlon, 9))[:, 0]
    ns = c["nstation"]
    if c["cap"]:  # 80% of the stations in 8 dense patches
        nl = ns * 4 // 5
        at = torch.randint(0, 8, (nl,), generator=g, device="cuda")
        plon, plat = _rand(g, 8, hi=360.0), torch.rad2deg(torch.asin(_rand(g, 8, lo=-0.8, hi=0.8)))
        slon = torch.cat([(plon[at] + 4.0 * _randn(g, nl)) % 360.0, _rand(g, ns - nl, hi=359.99)])
        slat = torch.cat([(plat[at] + 4.0 * _randn(g, nl)).clamp(-85, 85),
                          torch.rad2deg(torch.asin(_rand(g, ns - nl, lo=-1.0)))])
    else:
        slon, slat = _rand(g, ns, hi=359.99), torch.rad2deg(torch.asin(_rand(g, ns, lo=-1.0)))
    fi = slon / (360.0 / nlon)
    i0 = fi.floor().long() % nlon
    i1, ai = (i0 + 1) % nlon, fi - fi.floor()
    latt = torch.tensor(lat, device="cuda")
    j1 = torch.searchsorted(latt, slat).clamp(1, nlat - 1)
    j0 = j1 - 1
    aj = ((slat - latt[j0]) / (latt[j1] - latt[j0])).clamp(0.0, 1.0)

    def interp(f):  # (..., nlat, nlon) -> (..., ns)
        return (f[..., j0, i0] * (1 - ai) * (1 - aj) + f[..., j0, i1] * ai * (1 - aj) +
                f[..., j1, i0] * (1 - ai) * aj + f[..., j1, i1] * ai * aj)

    err = (1.0, 1.0, 1.0, 1.0e-4, 100.0)
    ps_at = interp(ps)                                     # (k + 1, ns)
    elm, lev, dat, er, hx = [], [], [], [], []
    for lv in np.unique(np.round(np.linspace(0, nlev - 1, c["obs_lev"])).astype(int)):
        for v, e in ((0, ID_U), (1, ID_V), (2, ID_T), (3, ID_Q)):
            y = interp(x3[v][:, lv])
            elm.append(torch.full((ns,), float(e), device="cuda", dtype=torch.float64))
            lev.append(sig_t[lv] * ps_at[k])
            dat.append(y[k] + err[v] * _randn(g, ns))
            er.append(torch.full_like(slon, err[v]))
            hx.append(y[:k])
    elm.append(torch.full((ns,), float(ID_PS), device="cuda", dtype=torch.float64))
    dat.append(ps_at[k] + err[4] * _randn(g, ns))
    lev.append(dat[-1])
    er.append(torch.full_like(slon, err[4]))
    hx.append(ps_at[:k])
    n = len(elm)
    return dict(lon=lon, lat=lat, sig=sig, x3=x3[:, :k].reshape(4, k, nlev, nlat * nlon),
                x2=ps[None, :k].reshape(1, k, nlat * nlon), elm=torch.cat(elm), olon=slon.repeat(n),
                olat=slat.repeat(n), lev=torch.cat(lev), dat=torch.cat(dat), err=torch.cat(er),
                hx=torch.cat(hx, dim=1))                   # hx (k, nobs)


def _regional_problem(c, seed):
    """u, v, w, T, qv, qr and pseudo-radar obs (Doppler and reflectivity buckets) on 60%
    of the columns at every level; perturbations and departures in obs space."""
    g = _gen(seed)
    nx, ny, nlev, k = c["nx"], c["ny"], c["nlev"], c["k"]
    zlev = (np.arange(nlev) + 0.5) * (15000.0 / nlev)
    amp = (10.0, 10.0, 2.0, 3.0, 2.0e-3, 1.0e-3)
    x3 = torch.empty((6, k, nlev, ny * nx), device="cuda", dtype=torch.float64)
    for v in range(6):
        f = (_waves(g, 1, nlev, ny, nx, 6) + 0.3 * _waves(g, k, nlev, ny, nx, 6, modes=4)) * amp[v]
        x3[v] = (f.abs() + 2.0e-4 if v == 5 else f).reshape(k, nlev, ny * nx)
    cols = torch.nonzero(_rand(g, ny * nx) < 0.6)[:, 0]
    lv = torch.arange(nlev, device="cuda").repeat_interleave(cols.numel())
    col = cols.repeat(nlev)
    n = col.numel()
    ri = ((col % nx) + 1 + _rand(g, n, lo=-0.5, hi=0.5)).clamp(1.0, nx)
    rj = (torch.div(col, nx, rounding_mode="floor") + 1 + _rand(g, n, lo=-0.5, hi=0.5)).clamp(1.0, ny)
    zt = torch.tensor(zlev, device="cuda")
    z = (zt[lv] + _rand(g, n, lo=-100.0, hi=100.0)).clamp(float(zlev[0]), float(zlev[-1]))
    bucket = (lv % 2).int()
    # Doppler: the wind towards a site south of the grid; reflectivity: 10 log10 of rain
    px, py = (ri - 1.0) * 500.0 - nx * 250.0, (rj - 1.0) * 500.0 + 20000.0
    rr = torch.sqrt(px * px + py * py)
    i0 = (ri - 1.0).floor().long().clamp(0, nx - 2)
    ai = ri - 1.0 - i0
    at = torch.div(col, nx, rounding_mode="floor") * nx + i0

    def interp(v):
        f = x3[v].reshape(k, -1)
        return f[:, lv * (ny * nx) + at] * (1 - ai) + f[:, lv * (ny * nx) + at + 1] * ai

    hx = torch.where(bucket == 0, (interp(0) * px + interp(1) * py) / rr,
                     10.0 * torch.log10(interp(5) * 1.0e5))
    hm = hx.mean(0)
    err = torch.where(bucket == 0, 3.0, 5.0).double()
    dep = hx.std(0) * _randn(g, n) + err * _randn(g, n)
    return dict(zlev=zlev, x3=x3, ri=ri, rj=rj, z=z, err=err, dep=dep, bucket=bucket,
                hd=hx - hm)                                # hd (k, nobs)


def _batch_problem(c, seed):
    """Obs table (nobs, k) with correlated rows, CSR lists of neighbouring obs and the
    background rows of the batch's points."""
    g = _gen(seed)
    npt, k, p, nobs = c["npt"], c["k"], min(c["p"], c["nobs"]), c["nobs"]
    hd = _randn(g, nobs, k) + 0.5 * _randn(g, nobs, 6) @ _randn(g, 6, k)
    hd -= hd.mean(1, keepdim=True)
    rd = _rand(g, nobs, lo=0.7, hi=3.0) ** 2
    dep = torch.sqrt(rd + 1.0) * _randn(g, nobs)
    cnt = torch.clamp(torch.round(p * _rand(g, npt, lo=0.2, hi=1.8)), 0, nobs).int()
    cnt[torch.randint(0, npt, (max(1, npt // 50),), generator=g, device="cuda")] = 0
    off = torch.zeros(npt + 1, dtype=torch.int64, device="cuda")
    off[1:] = torch.cumsum(cnt, 0)
    first = torch.randint(0, nobs, (npt,), generator=g, device="cuda")
    row = torch.repeat_interleave(torch.arange(npt, device="cuda"), cnt.long())
    idx = ((first[row] + torch.arange(row.numel(), device="cuda") - off[row]) % nobs).int()
    rho = torch.exp(-0.5 * _rand(g, row.numel(), hi=3.65) ** 2)
    infl = _rand(g, npt, lo=1.0, hi=1.2)
    xb = None
    if c["out"] == "apply":
        xb = 280.0 + 5.0 * _randn(g, npt, c["nv"], 1) + 2.0 * _randn(g, npt, c["nv"], k)
    return dict(hd=hd, rd=rd, dep=dep, cnt=cnt, off=off, idx=idx, rho=rho, infl=infl, xb=xb,
                row=row)


def _l96_problem(c, seed, k=None):
    g = _gen(seed)
    nx, k = c["nx"], k or c["k"]
    x = 8.0 + 0.1 * _randn(g, nx)

    def tend(s):
        return (torch.roll(s, -1) - torch.roll(s, 2)) * torch.roll(s, 1) - s + 8.0
    for _ in range(60):
        h = 0.01 * tend(x + 0.005 * tend(x))
        x = x + h
    xb = x[:, None] + _randn(g, nx, k)
    return dict(xb=xb, y=x + _randn(g, nx), gidx=np.arange(nx, dtype=np.int32), err=np.ones(nx))


class _View:
    """A handle's device array for torch, which keeps this object and so the handle alive."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f8", data=(ptr, False),
                                             version=2, strides=None)


def _analysis_views(h):
    """Torch views of the resident analysis: (points, variables, members) and, where the
    grid has 2-D variables, (columns, variables, members)."""
    p = [ctypes.c_void_p() for _ in range(4)]
    _lib.check(_lib.lib().lekf_device_state(h.h, *[ctypes.byref(q) for q in p]), "device_state")
    out = [torch.as_tensor(_View(h, p[1].value, (h.nij * h.nlev, h.nv3d, h.ne)), device="cuda")]
    if h.nv2d:
        out.append(torch.as_tensor(_View(h, p[3].value, (h.nij, h.nv2d, h.ne)), device="cuda"))
    return out


def _global_handle(c, q):
    h = GlobalLetkf(lon=q["lon"], lat=q["lat"], sig=q["sig"], ne=c["k"], sigma_obs=c["sigma"],
                    sigma_obsv=0.4, gross_error=10.0, prec=c["prec"], nobs_max=c["cap"],
                    q_top_lev=5 if c["nlev"] == 7 else 0, iq=3)
    h.set_ensemble(_host(q["x3"]), _host(q["x2"]))
    obs = [_host(q[n]) for n in ("elm", "olon", "olat", "lev", "dat", "err")]
    if not c["hx"]:
        h.set_obs(*obs, _host(q["hx"]))
    return h, obs


def prepare(case, seed):
    kind, c = case["kind"], case
    if kind == "core":
        q = _batch_problem(dict(npt=1, k=c["k"], p=c["p"], nobs=c["p"], out="core"), seed)
        return dict(kind=kind, c=c, hd=_host(q["hd"].T), rd=_host(q["rd"]), dep=_host(q["dep"]),
                    rho=np.exp(-0.5 * np.linspace(0.0, 3.0, c["p"]) ** 2))
    if kind == "batch":
        q = _batch_problem(c, seed)
        npt, k = c["npt"], c["k"]
        new = lambda *s: torch.zeros(s, device="cuda", dtype=torch.float64)  # noqa: E731
        out = dict(infl=new(npt), status=torch.zeros(npt, device="cuda", dtype=torch.int32))
        kw = {}
        if c["out"] == "trans":
            out.update(trans=new(npt, k, k), transm=new(npt, k), pao=new(npt, k, k))
            kw = dict(trans=out["trans"], transm=out["transm"], pao=out["pao"])
        else:
            out.update(xa=new(npt, c["nv"], k))
            kw = dict(apply=dict(nij=npt, nv3d=c["nv"], x3b=q["xb"], x3a=out["xa"]))
        job = make_job(k=k, npt=npt, hdxf=q["hd"], rdiag=q["rd"], dep=q["dep"], loc_off=q["off"],
                       loc_cnt=q["cnt"], loc_idx=q["idx"], loc_rho=q["rho"], infl_in=q["infl"],
                       infl_out=out["infl"], status=out["status"],
                       hdxf32=q["hd"].float() if c["prec"] != "f64" else None, **kw)
        return dict(kind=kind, job=job, prec=c["prec"], out=out)
    if kind == "l96":
        q = _l96_problem(c, seed)
        h = L96Letkf(nx=c["nx"], ne=c["k"], xlocal=3.0, infl_value=1.05)
        h.set_ensemble(_host(q["xb"].T.contiguous()[None, :, None, :]))
        return dict(kind=kind, h=h, y=_host(q["y"]), gidx=q["gidx"], err=q["err"])
    if kind == "global":
        h, obs = _global_handle(c, _global_problem(c, seed))
        if c["graph"]:
            h.set_graph(True)
        else:
            h.set_stream(torch.cuda.current_stream().cuda_stream)
        return dict(kind=kind, h=h, obs=obs if c["hx"] else None)
    if kind == "regional":
        q = _regional_problem(c, seed)
        h = RegionalLetkf(nx=c["nx"], ny=c["ny"], zlev=q["zlev"], dx=500.0, dy=500.0, ne=c["k"],
                          nv3d=6, sigma_h=c["sigma"], sigma_v=c["sigma"], nobs_max=c["cap"],
                          prec=c["prec"], infl_mode="fixed", infl_value=1.0)
        h.set_ensemble(_host(q["x3"]))
        h.set_obs(*[_host(q[n]) for n in ("ri", "rj", "z", "err", "dep", "bucket", "hd")])
        if c["relax"]:
            h.set_relax("rtps", c["relax"])
        h.set_stream(torch.cuda.current_stream().cuda_stream)
        return dict(kind=kind, h=h)
    hs = []
    for i, k in enumerate((c["k1"], c["k2"], c["k3"])):
        q = _l96_problem(c, seed + 1000 * i, k)
        h = L96Letkf(nx=c["nx"], ne=k, xlocal=3.0, infl_value=1.05)
        h.set_ensemble(_host(q["xb"].T.contiguous()[None, :, None, :]))
        h.set_obs(q["gidx"], _host(q["y"]), q["err"])
        hs.append(h)
    g = dict(c, k=c["kg"], obs_lev=c["nlev"], cap=0, prec="f64", sigma=500.0e3, hx=False)
    hs.append(_global_handle(g, _global_problem(g, seed))[0])
    return dict(kind=kind, hs=hs, stream=torch.cuda.current_stream().cuda_stream)


def run(state):
    s = state
    if s["kind"] == "core":
        c = s["c"]
        return letkf_core(c["k"], c["p"], c["p"], s["hd"], s["rd"], s["rho"], s["dep"], 1.05,
                          transm=True, pao=True)
    if s["kind"] == "batch":
        letkf_core_batch([s["job"]], s["prec"], torch.cuda.current_stream().cuda_stream)
        return s["out"]
    if s["kind"] == "l96":
        s["h"].set_obs(s["gidx"], s["y"], s["err"])
        s["h"].run()
        return _analysis_views(s["h"])
    if s["kind"] == "global":
        if s["obs"] is not None:
            s["h"].set_obs_hx(*s["obs"])
        s["h"].run()
        return _analysis_views(s["h"])
    if s["kind"] == "regional":
        s["h"].run()
        return _analysis_views(s["h"])
    run_batch(s["hs"], s["stream"])
    return [v for h in s["hs"] for v in _analysis_views(h)]


# --- what a pass cannot do without ------------------------------------------
def _point_work(npt, p, k, nv):
    """Gram of the smaller side (its symmetric half), its tridiagonal form and the rows of
    the state through it; the rows in and out."""
    m = min(p, k)
    flops = npt * (p * k * m + 4.0 * m ** 3 / 3.0 + 8.0 * (nv + 1) * k * m)
    return dict(flops=flops, bytes=npt * 16.0 * nv * k)


def work(case):
    c = case
    if c["kind"] == "core":
        w = _point_work(1, c["p"], c["k"], 0)
        return dict(flops=w["flops"] + 4.0 * c["k"] ** 3,
                    bytes=8.0 * (c["p"] * (c["k"] + 3) + 2 * c["k"] ** 2 + c["k"]))
    if c["kind"] == "batch":
        w = _point_work(c["npt"], c["p"], c["k"], c["nv"] if c["out"] == "apply" else 0)
        if c["out"] == "trans":
            w["flops"] += c["npt"] * 4.0 * c["k"] ** 3
            w["bytes"] += c["npt"] * 8.0 * (2 * c["k"] ** 2 + c["k"])
        w["bytes"] += 12.0 * c["npt"] * c["p"] + (8.0 if c["prec"] == "f64" else 4.0) * c["nobs"] * c["k"]
        return w
    if c["kind"] == "l96":
        w = _point_work(c["nx"], min(21, c["nx"]), c["k"], 1)
        return dict(w, bytes=w["bytes"] + 8.0 * c["nx"])
    if c["kind"] == "global":
        nobs = c["nstation"] * (4 * c["obs_lev"] + 1)
        p = nobs * min(1.0, (SPREAD * c["sigma"] / RE) ** 2 / 4.0) * (0.75 if c["nlev"] > 1 else 1.0)
        p = min(p, 0.5 * c["cap"]) if c["cap"] else p
        w = _point_work(c["nlon"] * c["nlat"] * c["nlev"], p, c["k"], 4)
        return dict(w, bytes=w["bytes"] + 8.0 * nobs * (6 + (0 if c["hx"] else c["k"])))
    if c["kind"] == "regional":
        n = c["nx"] * c["ny"]
        r = math.sqrt(CUT2) * c["sigma"]
        share = min(1.0, math.pi * (r / 500.0) ** 2 / n) * min(1.0, 1.3 * r / 15000.0)
        p = min(0.6 * n * c["nlev"] * share, 2.0 * c["cap"])
        w = _point_work(n * c["nlev"], p, c["k"], 6)
        return dict(w, bytes=w["bytes"] + 8.0 * 0.6 * n * c["nlev"] * (c["k"] + 5))
    w = [_point_work(c["nx"], 21, k, 1) for k in (c["k1"], c["k2"], c["k3"])]
    w.append(work(dict(c, kind="global", k=c["kg"], obs_lev=c["nlev"], cap=0, sigma=500.0e3, hx=False)))
    return dict(flops=sum(x["flops"] for x in w), bytes=sum(x["bytes"] for x in w))


# --- the same analyses in 64 bits --------------------------------------------
def _inv_sqrt(C):
    """C^-1/2 of a batch of positive definite matrices by the coupled Newton iteration."""
    s = C.abs().sum(2).amax(1)[:, None, None]
    eye = torch.eye(C.shape[1], device=C.device, dtype=C.dtype)
    Y, Z = C / s, eye.expand_as(C).contiguous()
    for _ in range(60):
        T = 1.5 * eye - 0.5 * (Z @ Y)
        if float((T - eye).abs().amax()) < 1e-13:
            break
        Y, Z = Y @ T, T @ Z
    return Z / torch.sqrt(s)


def _solve(W, hd, rd, dep, alpha):
    """Points with dense localisation weights W (n, nobs): Wa, w-bar, Pa and the adaptive
    inflation; a point without obs keeps sqrt(alpha) I."""
    n, k = W.shape[0], hd.shape[1]
    w = W / rd
    eye = torch.eye(k, device=W.device, dtype=W.dtype)
    C = torch.empty((n, k, k), device=W.device, dtype=W.dtype)
    for j in range(0, k, 16):
        yy = (hd[:, j:j + 16, None] * hd[:, None, :]).reshape(hd.shape[0], -1)
        C[:, j:j + 16] = (w @ yy).reshape(n, -1, k)
    p2 = C.diagonal(dim1=1, dim2=2).sum(1) / (k - 1)
    C = C + ((k - 1) / alpha)[:, None, None] * eye
    Z = _inv_sqrt(0.5 * (C + C.transpose(1, 2)))
    wa, pa = math.sqrt(k - 1) * Z, Z @ Z
    wm = (pa @ (w @ (hd * dep[:, None]))[:, :, None])[:, :, 0]
    p1, p3 = w @ (dep * dep), W.sum(1)
    q = (alpha * p2 + p3) / p2
    new = alpha + 0.0016 / (2.0 / p3 * q * q + 0.0016) * ((p1 - p3) / p2 - alpha)
    return wa, wm, pa, torch.where(p3 > 0, new, alpha)


def _apply(xb, wa, wm):
    xm = xb.mean(2, keepdim=True)
    return xm + (xb - xm) @ (wa + wm[:, :, None])


def _bin_count(c, q, ij, keep):
    """How often the search rectangle of columns ij covers each obs's lat band and lon cell
    (the reference's rectangle misses the sides of the cutoff disk near the poles)."""
    lon, lat = (torch.tensor(q[n], device="cuda") for n in ("lon", "lat"))
    olon, olat = q["olon"][keep], q["olat"][keep]

    def at(edges, x):
        return torch.searchsorted(edges.contiguous(), x.contiguous(), right=True) + 1
    band, cell = at(lat[1:-1], olat), at(lon[1:], olon)
    dlat = SPREAD * c["sigma"] / RE * 180.0 / math.pi
    lat1 = lat[torch.div(ij, c["nlon"], rounding_mode="floor")]
    lon1, dlon = lon[ij % c["nlon"]], dlat / torch.cos(lat1 * math.pi / 180.0)
    rows = ((band >= at(lat[1:-1], lat1 - dlat)[:, None]) &
            (band <= at(lat[1:-1], lat1 + dlat)[:, None]) & (olat >= lat[0]) & (olat < lat[-1]))
    lo = torch.where(dlon >= 180.0, 0.0, lon1 - dlon)
    hi = torch.where(dlon >= 180.0, 360.0, lon1 + dlon)
    below, above = lo < 0.0, hi > 360.0
    lo, hi = torch.where(below, lo + 360.0, lo), torch.where(above, hi - 360.0, hi)
    i0, i1 = at(lon[1:], lo), at(lon[1:], hi)
    wrap, both = below ^ above, below & above
    whole = ((lo < 0.0) | (hi > 360.0) | ((below & ~above) & (i0 < i1)) |
             ((above & ~below) & (i1 > i0)) | (both & (i0 > i1)))[:, None]
    ge, le = cell >= i0[:, None], cell <= i1[:, None]
    n = torch.where(wrap[:, None], ge.int() + le.int(), (ge & le).int())
    return torch.where(whole, 1, n) * rows


def _global_weights(c, q, b, keep):
    """Localisation weights of points b against the obs that pass the gross check."""
    nij = c["nlon"] * c["nlat"]
    ij, lev = b % nij, torch.div(b, nij, rounding_mode="floor")
    d2r = math.pi / 180.0
    lonp = torch.tensor(q["lon"], device="cuda")[ij % c["nlon"]] * d2r
    latp = torch.tensor(q["lat"], device="cuda")[torch.div(ij, c["nlon"], rounding_mode="floor")] * d2r
    lono, lato = q["olon"][keep] * d2r, q["olat"][keep] * d2r
    cosd = (torch.sin(lato) * torch.sin(latp)[:, None] + torch.cos(lato) *
            torch.cos(latp)[:, None] * torch.cos(lonp[:, None] - lono)).clamp(-1.0, 1.0)
    dist = torch.acos(cosd) * RE
    lnp = torch.log(q["x2"][0].mean(0)[ij] * torch.tensor(q["sig"], device="cuda")[lev])
    is_ps = q["elm"][keep] == ID_PS
    ln_o = torch.log(torch.where(is_ps, q["dat"][keep], q["lev"][keep]))
    dz = (ln_o - lnp[:, None]).abs()
    dz = torch.where(is_ps & (lev == 0)[:, None], 0.0, dz)
    rho = torch.exp(-0.5 * ((dist / c["sigma"]) ** 2 + (dz / 0.4) ** 2))
    rho = torch.where((dist <= SPREAD * c["sigma"]) & (dz <= SPREAD * 0.4), rho, 0.0)
    rho = rho * _bin_count(c, q, ij, keep)
    if c["cap"] and c["cap"] < rho.shape[1]:
        v, i = torch.topk(rho, c["cap"], dim=1)
        rho = torch.zeros_like(rho).scatter_(1, i, v)
    return rho


def _regional_weights(c, q, b):
    nij = c["nx"] * c["ny"]
    ij, lev = b % nij, torch.div(b, nij, rounding_mode="floor")
    dx = ((ij % c["nx"]) + 1.0)[:, None] - q["ri"]
    dy = (torch.div(ij, c["nx"], rounding_mode="floor") + 1.0)[:, None] - q["rj"]
    dz = torch.tensor(q["zlev"], device="cuda")[lev][:, None] - q["z"]
    nd = ((dx * 500.0) ** 2 + (dy * 500.0) ** 2 + dz * dz) / c["sigma"] ** 2
    rho = torch.where(nd <= CUT2, torch.exp(-0.5 * nd), 0.0)
    for u in (0, 1):
        at = torch.nonzero(q["bucket"] == u)[:, 0]
        if at.numel() > c["cap"]:
            v, i = torch.topk(rho[:, at], c["cap"], dim=1)
            rho[:, at] = torch.zeros((b.numel(), at.numel()), device="cuda",
                                     dtype=torch.float64).scatter_(1, i, v)
    return rho


def _grid_exact(c, x3, x2, hd, rd, dep, weights, infl, relax=0.0):
    """Analysis of every point, laid out as the handle keeps it."""
    nv, k, nlev, nij = x3.shape
    rows = x3.permute(2, 3, 0, 1).reshape(nlev * nij, nv, k)
    xa, xa2 = torch.empty_like(rows), None
    step = max(16, min(4096, int(2e9 / (8.0 * (rd.numel() + 3 * k * k)))))
    if x2 is not None:
        rows2 = x2.permute(2, 0, 1).contiguous()
        xa2 = torch.empty_like(rows2)
    for b0 in range(0, nlev * nij, step):
        b = torch.arange(b0, min(b0 + step, nlev * nij), device="cuda")
        wa, wm, _, _ = _solve(weights(b), hd, rd, dep,
                              torch.full((b.numel(),), infl, device="cuda", dtype=torch.float64))
        xa[b] = _apply(rows[b], wa, wm)
        if c["kind"] == "global" and nlev == 7:   # q keeps the background from level 5 up
            fixed = b >= 4 * nij
            xa[b[fixed], 3] = rows[b[fixed], 3]
        if x2 is not None and b0 < nij:
            s = b < nij
            xa2[b[s]] = _apply(rows2[b[s]], wa[s], wm[s])
    if relax:
        mb, ma = rows.mean(2, keepdim=True), xa.mean(2, keepdim=True)
        sb, sa = (rows - mb).std(2, keepdim=True), (xa - ma).std(2, keepdim=True)
        xa = ma + (xa - ma) * (relax * sb / sa - relax + 1.0)
    return [xa] if xa2 is None else [xa, xa2]


def _global_exact(c, seed):
    q = _global_problem(c, seed)
    hm = q["hx"].mean(0)
    dep = q["dat"] - hm
    keep = torch.nonzero(dep.abs() <= 10.0 * q["err"])[:, 0]
    return _grid_exact(c, q["x3"], q["x2"], (q["hx"] - hm).T[keep].contiguous(), q["err"][keep] ** 2,
                       dep[keep], lambda b: _global_weights(c, q, b, keep), 1.01)


def _l96_exact(c, seed, k=None):
    q = _l96_problem(c, seed, k)
    x = torch.arange(c["nx"], device="cuda", dtype=torch.float64)
    d = (x[:, None] - x).abs()
    d = torch.minimum(d, c["nx"] - d)
    rho = torch.exp(-0.5 * (d / 3.0) ** 2)
    rho = torch.where((d < SPREAD * 3.0) & (rho >= 1.0e-4), rho, 0.0)
    m = q["xb"].mean(1)
    return _grid_exact(c, q["xb"].T[None, :, None, :], None, q["xb"] - m[:, None],
                       torch.ones_like(m), q["y"] - m, lambda b: rho[b], 1.05)


def exact(case, seed):
    c = case
    if c["kind"] == "core":
        s = prepare(c, seed)
        t = [torch.tensor(np.ascontiguousarray(s[n])) for n in ("rho", "hd", "rd", "dep")]
        wa, wm, pa, a = _solve(t[0][None], *t[1:], torch.tensor([1.05], dtype=torch.float64))
        return wa[0], float(a[0]), wm[0], pa[0]
    if c["kind"] == "batch":
        q = _batch_problem(c, seed)
        out = dict(infl=[], status=None)
        for b0 in range(0, c["npt"], 1024):
            at = (q["row"] >= b0) & (q["row"] < b0 + 1024)
            W = torch.zeros((min(1024, c["npt"] - b0), c["nobs"]), device="cuda", dtype=torch.float64)
            W[q["row"][at] - b0, q["idx"][at].long()] = q["rho"][at]
            wa, wm, pa, a = _solve(W, q["hd"], q["rd"], q["dep"], q["infl"][b0:b0 + 1024])
            got = (dict(trans=wa, transm=wm, pao=pa) if c["out"] == "trans" else
                   dict(xa=_apply(q["xb"][b0:b0 + 1024], wa, wm)))
            for n, v in dict(got, infl=a).items():
                out.setdefault(n, []).append(v)
        return {n: v if v is None else torch.cat(v) for n, v in out.items()}
    if c["kind"] == "l96":
        return _l96_exact(c, seed)
    if c["kind"] == "global":
        npt, nobs = c["nlon"] * c["nlat"] * c["nlev"], c["nstation"] * (4 * c["obs_lev"] + 1)
        if c["hx"] or npt * (nobs * (c["k"] ** 2 + 50.0) + 80.0 * c["k"] ** 3) > 8e13:
            return None
        return _global_exact(c, seed)
    if c["kind"] == "regional":
        npt, nobs = c["nx"] * c["ny"] * c["nlev"], 0.6 * c["nx"] * c["ny"] * c["nlev"]
        if npt * (nobs * (c["k"] ** 2 + 1000.0) + 80.0 * c["k"] ** 3) > 3e13:
            return None
        q = _regional_problem(c, seed)
        return _grid_exact(c, q["x3"], None, q["hd"].T.contiguous(), q["err"] ** 2, q["dep"],
                           lambda b: _regional_weights(c, q, b), 1.0, c["relax"])
    out = []
    for i, k in enumerate((c["k1"], c["k2"], c["k3"])):
        out += _l96_exact(c, seed + 1000 * i, k)
    g = dict(c, kind="global", k=c["kg"], obs_lev=c["nlev"], cap=0, sigma=500.0e3, hx=False)
    return out + _global_exact(g, seed)
