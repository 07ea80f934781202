"""Badly conditioned points of the solve without eigenvalues (32 < k <= 95, no trans, no
pao): those past the rational form's tables are listed and solved by the fused eigen
kernel, all at once, and agree with it in every precision.

Timings compare batches within one process and with wide margins: 256 listed points run
on 256 CUs in about the time of one (one after another they took 64 times it).
"""
import time

import numpy as np
import pytest

import oracle
from letkf_amd import _lib, core, tune
from letkf_amd.device import DeviceArray, sync

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.fixture
def knobs():
    before = tune.current()
    yield
    for name, v in before.items():
        tune.set(name, v)


def _problem(k, spreads, p, seed, nv=4):
    rng = np.random.default_rng(seed)
    npt = len(spreads)
    n = npt * p
    hd = rng.standard_normal((n, k)) * np.repeat(spreads, p)[:, None]
    hd -= hd.mean(axis=1, keepdims=True)
    return dict(k=k, npt=npt, nv=nv, hd=hd, rd=rng.uniform(0.5, 2.0, n), dep=rng.standard_normal(n),
                rho=rng.uniform(0.1, 1.0, n), off=np.arange(npt + 1, dtype=np.int64) * p,
                xb=rng.standard_normal((npt, nv, k)))


def _job(q, prec="f64"):
    t = DeviceArray.from_numpy
    k, npt, nv = q["k"], q["npt"], q["nv"]
    out = dict(xa=DeviceArray.zeros((npt, nv, k)), transm=DeviceArray.zeros((npt, k)),
               status=DeviceArray.zeros((npt,), np.int32), infl=DeviceArray.zeros(npt))
    kw = {"hdxf32": t(q["hd"].astype(np.float32))} if prec != "f64" else {}
    job = core.make_job(k=k, npt=npt, hdxf=t(q["hd"]), rdiag=t(q["rd"]), dep=t(q["dep"]),
                        loc_off=t(q["off"]), loc_idx=t(np.arange(q["hd"].shape[0], dtype=np.int32)),
                        loc_rho=t(q["rho"]), infl_in=t(np.full(npt, 1.05)), infl_out=out["infl"],
                        status=out["status"], transm=out["transm"],
                        apply=dict(nij=npt, nv3d=nv, nv2d=0, x3b=t(q["xb"]), x3a=out["xa"]), **kw)
    return job, out


def _kappa(q, b):
    sl = slice(q["off"][b], q["off"][b + 1])
    c = (q["hd"][sl].T * (q["rho"][sl] / q["rd"][sl])) @ q["hd"][sl]
    lam = np.linalg.eigvalsh(c + (q["k"] - 1) / 1.05 * np.eye(q["k"]))
    return lam[-1] / lam[0]


def _ms(job, prec="f64"):
    ts = []
    for i in range(6):
        sync()
        t0 = time.perf_counter()
        core.letkf_core_batch([job], prec)
        sync()
        ts.append(time.perf_counter() - t0)
    return 1e3 * min(ts[1:])


@pytest.mark.parametrize("k", [40, 64, 80])
def test_listed_points_run_side_by_side(gpu, k):
    """Past the truncation threshold every point is listed: 256 of them against one."""
    one, _ = _job(_problem(k, [1e5], 2 * k, 1))
    many, out = _job(_problem(k, [1e5] * 256, 2 * k, 1))
    t1, tn = _ms(one), _ms(many)
    print(f"k={k}: 1 point {t1:.3f} ms, 256 points {tn:.3f} ms", flush=True)
    assert (out["status"].numpy() & _lib.LEKF_PT_RANKDEF).all()
    assert tn < 8 * t1


@pytest.mark.parametrize("k,nv", [(40, 5), (64, 9), (80, 3), (120, 2), (200, 6)])
def test_tables_reach_the_truncation_threshold(gpu, k, nv):
    """Condition numbers from 2^20 to the truncation threshold 2^26 (common_mtx.f90:66-74):
    the rational form's, without eigenvalues, as fast as well conditioned points, against
    oracle.letkf_core.  Both sides are backward stable: a small multiple of k eps cond(A)."""
    q = _problem(k, [700.0, 1500.0, 2500.0, 3000.0], 2 * k, k, nv)
    job, out = _job(q)
    core.letkf_core_batch([job])
    sync()
    a = {n: x.numpy() for n, x in out.items()}
    kaps = []
    for b in range(q["npt"]):
        sl = slice(q["off"][b], q["off"][b + 1])
        ref = oracle.letkf_core(q["hd"][sl], q["rd"][sl], q["rho"][sl], q["dep"][sl], 1.05,
                                transm=True)
        kap = _kappa(q, b)
        kaps.append(kap)
        tol = 8 * k * EPS * kap
        xm = q["xb"][b].mean(axis=1, keepdims=True)
        want = xm + (q["xb"][b] - xm) @ (ref["trans"] + ref["transm"][:, None])
        assert a["status"][b] == 0
        assert np.abs(a["xa"][b] - want).max() <= tol * np.abs(want - xm).max() + 1e-13
        assert np.abs(a["transm"][b] - ref["transm"]).max() <= tol * np.abs(ref["transm"]).max()
    assert 2 ** 20 < min(kaps) and max(kaps) < 2 ** 26, kaps
    hard, easy = (_job(_problem(k, [s] * 256, 2 * k, 3, nv))[0] for s in (1500.0, 0.5))
    th, te = _ms(hard), _ms(easy)
    print(f"k={k}: condition {min(kaps):.2g} .. {max(kaps):.2g}, {th:.3f} ms, {te:.3f} ms well conditioned",
          flush=True)
    assert th < 3 * te


def test_large_k_past_the_tables(gpu):
    """k = 200 past the truncation threshold: QL runs on one of a point's four waves, and
    two points share a CU where one wave per point left room for four.  With the rotations
    applied in the recurrence's shadow a point takes 4.0 times a well conditioned one's
    time, as long as one wave per point took; with a sweep's rotations applied after it 5.4."""
    hard, easy = (_job(_problem(200, [s] * 1024, 220, 3))[0] for s in (1e5, 0.5))
    th, te = _ms(hard), _ms(easy)
    print(f"k=200: {th:.2f} ms, {te:.2f} ms well conditioned", flush=True)
    assert th < 4.7 * te


@pytest.mark.parametrize("k", [36, 40, 57, 64])
def test_mixed_forms_past_their_tables(gpu, knobs, k):
    """FP32 and split-BF16x3 without the FP64 redo: condition numbers below and above the
    mixed forms' last table (4 * 8^4), against the fused kernel on the same Gram.  Both are
    backward stable: a small multiple of k eps cond(A)."""
    _mixed(k)


@pytest.mark.parametrize("k", [65, 72, 80, 95])
def test_mixed_forms_past_their_tables_lds(gpu, knobs, k):
    _mixed(k)


def _mixed(k):
    tune.set("mixed_kappa", 0)
    q = _problem(k, [0.2, 1.0, 4.0, 12.0, 25.0, 40.0, 80.0], 2 * k, k)
    kap = np.array([_kappa(q, b) for b in range(q["npt"])])
    assert kap.min() < 32 and (kap < 16384).sum() >= 4 and (kap > 16384).sum() >= 1
    for prec in ("f32", "bf16x3"):
        res = []
        for split in (1, 0):
            tune.set("eig_split", split)
            job, out = _job(q, prec)
            core.letkf_core_batch([job], prec)
            sync()
            res.append({n: a.numpy() for n, a in out.items()})
        a, f = res
        np.testing.assert_array_equal(a["status"], f["status"])
        for b in range(q["npt"]):
            tol = 8 * k * EPS * kap[b]
            for n in ("xa", "transm"):
                d = np.abs(a[n][b] - f[n][b]).max()
                assert d <= tol * np.abs(f[n][b]).max(), (prec, b, kap[b], n, d)
            assert abs(a["infl"][b] - f["infl"][b]) <= 1e-12 * abs(f["infl"][b]), (prec, b)


@pytest.mark.parametrize("k", [33, 40, 64])
@pytest.mark.parametrize("prec,thr", [("f32", 125), ("bf16x3", 2000)])
def test_redo_list_at_its_edge(gpu, knobs, k, prec, thr):
    """The FP64 redo of a plain job first bounds the condition number by lambda_max over
    0.75 (k-1)/infl and takes the extreme eigenvalues only where that passes.  Points of
    one mode (lambda_min is (k-1)/infl itself) around that bound and around the threshold
    (2000; FP32 takes 16 times the value set), and points far past the bound whose smallest
    eigenvalue is large too: the ones above the threshold get the FP64 solve's bits, the
    others the plain mixed solve's.  2% off the threshold is 20 times what the mixed
    Gram (5e-7 of lambda_max) moves lambda_min there."""
    eff, rng = 2000.0, np.random.default_rng(k)
    goal = eff * np.array([0.5, 0.74, 0.76, 0.98, 1.02, 1.3, 1.36, 6.0, 0.0, 0.0, 0.0])
    p = 4 * k
    q = _problem(k, [1.0] * goal.size, p, k)
    for b in range(goal.size):
        sl = slice(b * p, (b + 1) * p)
        if not goal[b]:  # of full rank: the members' mean is left in
            q["hd"][sl] = 30.0 * rng.standard_normal((p, k))
            continue
        v = rng.standard_normal(k)
        q["hd"][sl] = np.outer(rng.standard_normal(p), v - v.mean())
        q["hd"][sl] *= np.sqrt((goal[b] - 1.0) / (_kappa(q, b) - 1.0))
    kap = np.array([_kappa(q, b) for b in range(q["npt"])])
    above = kap > eff
    np.testing.assert_allclose(kap[goal > 0], goal[goal > 0], rtol=1e-6)
    assert above.sum() == 4 and kap[goal == 0].max() < 0.1 * eff

    def run(prec, value):
        tune.set("mixed_kappa", value)
        job, out = _job(q, prec)
        core.letkf_core_batch([job], prec)
        sync()
        return {n: a.numpy() for n, a in out.items()}

    ref, mix, got = run("f64", thr), run(prec, 0), run(prec, thr)
    np.testing.assert_array_equal((got["status"] & _lib.LEKF_PT_FP64) != 0, above)
    for n in ("xa", "transm", "infl"):
        np.testing.assert_array_equal(got[n][above], ref[n][above])
        np.testing.assert_array_equal(got[n][~above], mix[n][~above])
