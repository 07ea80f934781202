"""The regional cap's blocks (reg_select_wave): caps at the edges of its chunks of 64 and
blocks of 224 and at the ends of its range, equal keys across blocks, errors spread over
decades, obs within rounding of the cutoff, and coordinates that FP32 resolves coarsely.

Reference: the uncapped lists of the same obs (another kernel: scan order, rho in FP64)
through the oracle's cap, keys err^2 / rho.  Equal entry by entry: set, slot order, rho.
"""
import numpy as np
import pytest

import oracle
from letkf_amd import das

pytestmark = pytest.mark.gpu

NX, NY, NLEV, DX, SIG = 20, 16, 4, 500.0, 1500.0


def _obs(kind, seed, nbkt):
    rng = np.random.default_rng(seed)
    z0 = 9.0e4 if kind == "coarse" else 0.0
    zlev = z0 + 1000.0 + 2500.0 * np.arange(NLEV)
    n = 12 * NX * NY * NLEV
    ri, rj = rng.uniform(0.5, NX + 0.5, n), rng.uniform(0.5, NY + 0.5, n)
    z = rng.uniform(zlev[0] - 500.0, zlev[-1] + 500.0, n)
    err = np.full(n, 3.0)
    if kind == "errors":
        err = np.exp(rng.normal(0.0, 2.0, n))
        err[:20] = 0.0
    if kind == "ties":
        at = rng.choice(n, 900, replace=False)
        ri[at], rj[at], z[at] = 10.25, 8.25, zlev[1]
    if kind == "cutoff":
        # a ring around column (10, 8): distances within 1e-4 .. 1e-15 of the cutoff
        m = 600
        r = np.sqrt(13.33333333) * SIG / DX * (1.0 + rng.choice([-1, 1], m) *
                                               10.0 ** rng.uniform(-15, -4, m))
        a = rng.uniform(0.0, 2.0 * np.pi, m)
        ri[:m], rj[:m], z[:m] = 10.0 + r * np.cos(a), 8.0 + r * np.sin(a), zlev[2]
    return dict(ri=ri, rj=rj, z=z, err=err, bucket=rng.integers(0, nbkt, n).astype(np.int32),
                zlev=zlev)


def _handle(o, cap, rng):
    h = das.RegionalLetkf(nx=NX, ny=NY, zlev=o["zlev"], dx=DX, dy=DX, ne=4, nv3d=1, sigma_h=SIG,
                          sigma_v=SIG, nobs_max=cap, infl_value=1.0)
    h.set_ensemble(rng.standard_normal((NX * NY, NLEV, 4, 1)))
    n = o["ri"].size
    h.set_obs(o["ri"], o["rj"], o["z"], o["err"], np.zeros(n), o["bucket"], np.zeros((n, 4)))
    h.select()
    h.sync()
    return h


@pytest.mark.parametrize("cap,kind,nbkt", [(1, "plain", 2), (63, "plain", 1), (64, "ties", 2),
                                           (65, "errors", 3), (223, "plain", 4), (224, "errors", 2),
                                           (225, "ties", 1), (448, "cutoff", 2), (700, "ties", 2),
                                           (1000, "coarse", 1), (1023, "cutoff", 1),
                                           (1024, "errors", 1), (1024, "plain", 4)])
def test_cap_blocks(gpu, cap, kind, nbkt):
    o = _obs(kind, 1000 + cap, nbkt)
    rng = np.random.default_rng(cap)
    h, h0 = _handle(o, cap, rng), _handle(o, 0, rng)
    perm, _ = h.obs_index()
    err, bkt = o["err"][perm], o["bucket"][perm]
    pts = rng.choice(NX * NY * NLEV, 60, replace=False).tolist() + [2 * NX * NY + 7 * NX + 9]
    bound = 0
    for b in pts:
        idx, rho = h.local(b)
        full, frho = h0.local(b)
        want = []
        for t in range(nbkt):
            sel = np.flatnonzero(bkt[full] == t)
            if sel.size > cap:
                sel = sel[oracle.cap_stream(err[full[sel]] ** 2 / frho[sel], cap)]
                bound += 1
            want.append(sel)
        want = np.concatenate(want)
        np.testing.assert_array_equal(idx, full[want])
        np.testing.assert_array_equal(rho, frho[want])
    h.close()
    h0.close()
    if cap < 900:
        assert bound > 0
