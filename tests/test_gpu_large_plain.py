"""The local solve of k > 95 without trans and pao outputs: both forms (0 < p < k and
p >= k) at the edges of their 64-element blocks and rows of eight, points without obs,
condition numbers from 1 through every table of the rational form to past the last one
(solved by QL), more state rows than one pass takes.  Against oracle.letkf_core + apply.

Tolerance: both sides are backward stable, so the functions of A agree to a small
multiple of k eps cond(A), relative to the largest analysis increment or perturbation
of the point's rows, plus the rounding of the rows' means.
"""
import numpy as np
import pytest

import oracle
from letkf_amd import _lib, core
from letkf_amd.device import DeviceArray, sync

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.mark.parametrize("k,nv", [(96, 1), (97, 16), (127, 9), (128, 3), (130, 7), (192, 2),
                                  (200, 5), (255, 16), (256, 8)])
def test_large_plain_matches_oracle(gpu, k, nv):
    rng = np.random.default_rng(100 * k + nv)
    sizes = [0, 1, 2, 3, 7, 64, 65, k - 1, k, k + 70]
    spreads = [1e-6, 0.3, 2.0, 8.0, 30.0, 100.0, 400.0, 4e4]
    pts = [(p, spreads[(i + j) % len(spreads)]) for i, p in enumerate(sizes) for j in (0, 3, 6)]
    pts += [(p, s) for p in (64, k + 70) for s in spreads]
    npt = len(pts)
    cnt = np.array([p for p, _ in pts], np.int32)
    off = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int64)
    n = int(off[-1])
    hd = rng.standard_normal((n, k)) * np.repeat([s for _, s in pts], cnt)[:, None]
    hd -= hd.mean(axis=1, keepdims=True)
    rd = rng.uniform(0.5, 2.0, n)
    dep = rng.standard_normal(n)
    rho = rng.uniform(0.05, 1.0, n)
    infl = rng.uniform(1.0, 1.2, npt)
    xb = 250.0 + rng.standard_normal((npt, nv, k)) * 3.0

    d = {m: DeviceArray.from_numpy(v) for m, v in
         dict(hd=hd, rd=rd, dep=dep, off=off, cnt=cnt, idx=np.arange(n, dtype=np.int32), rho=rho,
              infl=infl, xb=xb).items()}
    xa, inf2, wm, st = (DeviceArray.zeros(s, t) for s, t in
                        ((xb.shape, np.float64), (npt, np.float64), ((npt, k), np.float64),
                         (npt, np.int32)))
    kw = dict(k=k, npt=npt, hdxf=d["hd"], rdiag=d["rd"], dep=d["dep"], loc_off=d["off"],
              loc_cnt=d["cnt"], loc_idx=d["idx"], loc_rho=d["rho"], infl_in=d["infl"],
              infl_out=inf2, status=st, transm=wm)
    # the second job of the launch outputs trans: the two kernels share the launch
    tr = DeviceArray.zeros((1, k, k), np.float64)
    sel = pts.index((k + 70, 30.0), npt - len(spreads))
    one = {m: DeviceArray.from_numpy(v) for m, v in
           dict(off=off[sel:sel + 2].copy(), infl=infl[sel:sel + 1].copy(),
                inf2=np.zeros(1)).items()}
    core.letkf_core_batch([
        core.make_job(apply=dict(nij=npt, nv3d=nv, nv2d=0, x3b=d["xb"], x3a=xa), **kw),
        core.make_job(k=k, npt=1, hdxf=d["hd"], rdiag=d["rd"], dep=d["dep"], loc_off=one["off"],
                      loc_idx=d["idx"], loc_rho=d["rho"], infl_in=one["infl"],
                      infl_out=one["inf2"], trans=tr)])
    sync()
    a, i2, w2, s2 = xa.numpy(), inf2.numpy(), wm.numpy(), st.numpy()

    levels = set()
    for b, (p, s) in enumerate(pts):
        sl = slice(off[b], off[b + 1])
        ref = oracle.letkf_core(hd[sl], rd[sl], rho[sl], dep[sl], infl[b], transm=True)
        C = (hd[sl].T * (rho[sl] / rd[sl])) @ hd[sl] + (k - 1) / infl[b] * np.eye(k)
        lam = np.linalg.eigvalsh(C)
        kap = lam[-1] / lam[0]
        levels.add(int(np.ceil(np.log2(max(kap, 1.0)) / 3)))
        tol = 8 * k * EPS * kap
        assert bool(s2[b] & _lib.LEKF_PT_RANKDEF) == (kap > 1.0 / np.sqrt(EPS)), (p, s, kap)
        assert not s2[b] & _lib.LEKF_PT_NOCONV, (p, s, kap)
        if kap > 1.0 / np.sqrt(EPS):
            assert np.isfinite(a[b]).all()
            continue
        xm = xb[b].mean(axis=1, keepdims=True)
        want = xm + (xb[b] - xm) @ (ref["trans"] + ref["transm"][:, None])
        scale = np.abs(want - xm).max()
        assert np.abs(a[b] - want).max() <= tol * scale + 2 * k * EPS * np.abs(xm).max(), (p, s, kap)
        assert np.abs(w2[b] - ref["transm"]).max() <= tol * np.abs(ref["transm"]).max(), (p, s, kap)
        if b == sel:  # the second job: trans (column-major) with w-bar in it
            full = ref["trans"] + ref["transm"][:, None]
            assert np.abs(tr.numpy()[0].T - full).max() <= tol * np.abs(full).max(), kap
            assert abs(one["inf2"].numpy()[0] - ref["parm_infl"]) <= tol * abs(ref["parm_infl"])
        if p:
            assert abs(i2[b] - ref["parm_infl"]) <= 1e-12 * abs(ref["parm_infl"]) + tol
        else:
            assert i2[b] == infl[b]
    assert len(levels) >= 6  # condition numbers across the tables
