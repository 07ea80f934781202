"""Jobs of different ensemble sizes and outputs in one batch (32 < k <= 95): jobs of one
kernel class share the solve's launches, the Gram taking one launch per column cut, and
jobs with and without trans share records, flags and the FP64 redo list.  Every job's
outputs equal, bit for bit, those of the same job launched alone.
"""
import numpy as np
import pytest

from letkf_amd import _lib, core, device, tune
from letkf_amd.device import DeviceArray, sync

pytestmark = pytest.mark.gpu

SIZES = [0, 1, 5, 64, 130, 33, 200]


@pytest.fixture
def knobs():
    before = tune.current()
    yield
    for name, v in before.items():
        tune.set(name, v)


def _job(k, trans, seed, prec, nv=3):
    rng = np.random.default_rng(seed)
    cnt = np.array([SIZES[(i + seed) % len(SIZES)] for i in range(2 * len(SIZES))])
    off = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int64)
    n, npt = int(off[-1]), cnt.size
    # the points alternate between well and badly conditioned
    scale = np.repeat(np.where(np.arange(npt) % 2, 4.0, 0.3), cnt)
    hd = rng.standard_normal((n, k)) * scale[:, None]
    hd -= hd.mean(axis=1, keepdims=True)
    t = DeviceArray.from_numpy
    out = dict(infl=DeviceArray.zeros(npt), status=DeviceArray.zeros((npt,), np.int32),
               transm=DeviceArray.zeros((npt, k)), xa=DeviceArray.zeros((npt, nv, k)))
    kw = {}
    if trans:
        out["trans"] = kw["trans"] = DeviceArray.zeros((npt, k, k))
    if prec != "f64":
        kw["hdxf32"] = t(hd.astype(np.float32))
    job = core.make_job(k=k, npt=npt, hdxf=t(hd), rdiag=t(rng.uniform(0.5, 2.0, n)),
                        dep=t(rng.standard_normal(n)), loc_off=t(off),
                        loc_idx=t(np.arange(n, dtype=np.int32)),
                        loc_rho=t(rng.uniform(0.1, 1.0, n)), infl_in=t(rng.uniform(1.0, 1.2, npt)),
                        infl_out=out["infl"], status=out["status"], transm=out["transm"],
                        apply=dict(nij=npt, nv3d=nv, nv2d=0,
                                   x3b=t(rng.standard_normal((npt, nv, k))), x3a=out["xa"]), **kw)
    return job, out


def _run(specs, prec, together):
    js = [_job(k, tr, 7 * i + k, prec) for i, (k, tr) in enumerate(specs)]
    if together:
        core.letkf_core_batch([j for j, _ in js], prec)
        sync()
    else:
        for j, _ in js:
            core.letkf_core_batch([j], prec)
            sync()
    return [{n: a.numpy() for n, a in out.items()} for _, out in js]


@pytest.mark.parametrize("prec", ["f64", "bf16x3"])
@pytest.mark.parametrize("specs", [[(40, False), (40, True)],
                                   [(40, False), (47, False)], [(50, False), (52, False), (51, False)],
                                   [(33, True), (36, False), (40, True), (47, False), (48, True)],
                                   [(49, False), (57, True), (63, False), (64, True)],
                                   [(64, False), (64, True), (65, True), (67, False)],
                                   [(65, False), (72, True), (78, False), (80, True)],
                                   [(81, True), (90, False), (95, True)]])
def test_job_alone_equals_job_in_batch(gpu, knobs, specs, prec):
    if prec != "f64":
        tune.set("mixed_kappa", 30)
    alone, batch = _run(specs, prec, False), _run(specs, prec, True)
    for (k, tr), a, b in zip(specs, alone, batch):
        for name in a:
            np.testing.assert_array_equal(a[name], b[name], err_msg=f"k={k} trans={tr} {name}")
        redone = (b["status"] & _lib.LEKF_PT_FP64) != 0
        assert redone.any() == (prec != "f64" and k <= 64), (k, tr)
        assert not redone.all()


@pytest.mark.parametrize("ks", [range(33, 48), range(48, 65)])
def test_one_solve_launch_per_class(gpu, ks):
    """Trans jobs of one class: one tridiagonalisation, QL and apply for all of them, and
    one Gram launch per cut of the columns."""
    js = [_job(k, True, k, "f64") for k in ks]
    sync()
    device.ktime_enable(True)
    core.letkf_core_batch([j for j, _ in js], "f64")
    sync()
    kt = device.ktime_all()
    device.ktime_enable(False)
    assert {n: kt[n][1] for n in ("eig_tri", "eig_ql", "eig_apply")} == \
        {"eig_tri": 1, "eig_ql": 1, "eig_apply": 1}
    assert 1 <= kt["gram"][1] <= 4  # k + 1 = 33 .. 48 or 49 .. 65 columns: three or four cuts
