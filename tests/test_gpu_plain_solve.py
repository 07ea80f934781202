"""The eigenvalue-free local solve (32 < k <= 95, jobs without trans and pao) at the
edges of its register tiles: k around multiples of 8, one to three groups of eight rows
(state rows + b), points without obs, with one obs, with p < k and p > k, and condition
numbers from 1 through every table of the rational form to past the last one (left to
the eigenvector kernel).  Against oracle.letkf_core + apply.

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


@pytest.mark.parametrize("k,nv", [(33, 1), (40, 7), (41, 8), (48, 16), (49, 3), (56, 6), (57, 7),
                                  (64, 15), (65, 2), (72, 7), (73, 8), (80, 5), (88, 7), (95, 16)])
def test_plain_solve_matches_oracle(gpu, k, nv):
    rng = np.random.default_rng(100 * k + nv)
    sizes = [0, 1, k // 2, k, k + 5, 3 * k]
    spreads = [1e-6, 0.3, 2.0, 8.0, 30.0, 100.0, 400.0, 4e4]
    pts = [(p, s) for p in sizes for s in spreads]
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
              infl_out=inf2, status=st,
              apply=dict(nij=npt, nv3d=nv, nv2d=0, x3b=d["xb"], x3a=xa))
    core.letkf_core_batch([core.make_job(**kw)])
    sync()
    a, i2, s2 = xa.numpy(), inf2.numpy(), st.numpy()
    # the same points with the mean weights asked for: Wa alone is applied
    core.letkf_core_batch([core.make_job(transm=wm, **kw)])
    sync()
    w2 = wm.numpy()

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
        if kap > 1.0 / np.sqrt(EPS):
            assert np.isfinite(a[b]).all()
            continue
        xm = xb[b].mean(axis=1, keepdims=True)
        want = xm + (xb[b] - xm) @ (ref["trans"] + ref["transm"][:, None])
        scale = np.abs(want - xm).max()
        assert np.abs(a[b] - want).max() <= tol * scale + 2 * k * EPS * np.abs(xm).max(), (p, s, kap)
        assert np.abs(w2[b] - ref["transm"]).max() <= tol * np.abs(ref["transm"]).max(), (p, s, kap)
        if p:
            assert abs(i2[b] - ref["parm_infl"]) <= 1e-12 * abs(ref["parm_infl"]) + tol
        else:
            assert i2[b] == infl[b]
    assert len(levels) >= 6  # condition numbers across the tables
