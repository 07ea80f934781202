"""The FP64 Gram of 32 < k <= 95 at every cut of its columns (full 16-column tiles, then
strips of four: k + 1 at and around multiples of 4 and 16), for list lengths around the
4-obs steps, the chunks of 64 and the waves' turns.

The analysis with obs perturbations member by member (y_so = 1) takes the same sums in
the same order as row by row, so it is bit-identical; transm against oracle.letkf_core
with the bound of two backward stable solves, a small multiple of k eps cond(A), plus
the sums' (p + k) eps.
"""
import numpy as np
import pytest

import oracle
from letkf_amd import core
from letkf_amd.device import DeviceArray, sync

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps
SIZES = [1, 3, 4, 5, 63, 64, 65, 67, 68, 128, 129, 191, 257, 517]


@pytest.mark.parametrize("k", [33, 35, 36, 38, 39, 40, 43, 47, 50, 51, 52, 55, 56, 60, 63, 64, 67,
                               71, 79, 80, 83, 87, 88, 92, 95])
def test_gram_columns(gpu, k):
    rng = np.random.default_rng(k)
    npt = len(SIZES)
    off = np.concatenate([[0], np.cumsum(SIZES)]).astype(np.int64)
    n = int(off[-1])
    hd = rng.standard_normal((n, k))
    hd -= hd.mean(axis=1, keepdims=True)
    rd, dep, rho = rng.uniform(0.5, 2.0, n), rng.standard_normal(n), rng.uniform(0.05, 1.0, n)
    idx = np.concatenate([rng.permutation(n)[:p] for p in SIZES]).astype(np.int32)
    ones = np.ones(npt)
    d = {m: DeviceArray.from_numpy(v) for m, v in
         dict(rows=hd, cols=np.ascontiguousarray(hd.T), rd=rd, dep=dep, off=off, idx=idx, rho=rho,
              infl=ones).items()}
    out = []
    for name, strides in (("rows", {}), ("cols", dict(y_so=1, y_sm=n))):
        wm = DeviceArray.zeros((npt, k), np.float64)
        inf2 = DeviceArray.zeros(npt, np.float64)
        core.letkf_core_batch([core.make_job(
            k=k, npt=npt, hdxf=d[name], rdiag=d["rd"], dep=d["dep"], loc_off=d["off"],
            loc_idx=d["idx"], loc_rho=d["rho"], infl_in=d["infl"], infl_out=inf2, transm=wm,
            apply=dict(nij=npt, nv3d=1, nv2d=0, x3b=_xb(npt, k),
                       x3a=DeviceArray.zeros((npt, 1, k), np.float64)), **strides)])
        sync()
        out.append((wm.numpy(), inf2.numpy()))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
    for b, p in enumerate(SIZES):
        o, r = idx[off[b]:off[b + 1]], rho[off[b]:off[b + 1]]
        ref = oracle.letkf_core(hd[o], rd[o], r, dep[o], 1.0, transm=True)
        lam = np.linalg.eigvalsh((hd[o].T * (r / rd[o])) @ hd[o] + (k - 1) * np.eye(k))
        tol = (8 * k + p + k) * EPS * lam[-1] / lam[0]
        assert np.abs(out[0][0][b] - ref["transm"]).max() <= tol * np.abs(ref["transm"]).max(), p
        assert abs(out[0][1][b] - ref["parm_infl"]) <= tol * abs(ref["parm_infl"]), p


def _xb(npt, k):
    return DeviceArray.from_numpy(np.random.default_rng(0).standard_normal((npt, 1, k)))
