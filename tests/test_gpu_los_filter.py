"""The on-sky (rp, pi) pair filter's line-of-sight test against the oracle where its bounds are
weakest: around the observer (|x_i + x_j| down to 0, |l|^2 below the 3-D limit), far away (FP32
squares of large distances), separations on the rp and pi limits, wide and narrow windows. The
filter may only drop pairs that the FP64 decision rejects, so the counts are equal."""
import os

import numpy as np
import pytest

from corrfunc_amd import _abi, _lib

from test_gpu_mocks import assert_same, bins_file, opts

pytestmark = pytest.mark.gpu


def _catalog(kind, n, rng, rpmax):
    if kind == "observer":      # all around the origin, out to twice the separations
        ra, dec = rng.uniform(0, 360, n), np.degrees(np.arcsin(rng.uniform(-1, 1, n)))
        return [ra, dec, 60.0 * np.cbrt(rng.uniform(0, 1, n)) + 1e-3]
    if kind == "far":           # a narrow beam at thousands of Mpc/h
        return [rng.uniform(100, 101.2, n), rng.uniform(20, 21.2, n), rng.uniform(3000, 3080, n)]
    # "limits": pairs whose transverse separation lies within quanta of rpmax
    d = rng.uniform(180, 240, n)
    dec = np.degrees(rng.choice([0.0, rpmax / 210.0], n) + rng.normal(0, 1e-4, n))
    return [rng.uniform(150, 156, n), dec + 10.0, d]


@pytest.mark.parametrize("dense", ["0", "2"])
@pytest.mark.parametrize("kind", ["observer", "far", "limits"])
@pytest.mark.parametrize("rpmax,pimax", [(20.0, 30.0), (30.0, 5.0), (6.0, 40.0)])
def test_filter_keeps_every_pair(engine, oracle, tmp_path, kind, rpmax, pimax, dense):
    os.environ["CORRFUNC_AMD_DENSE"] = dense
    _lib.set_engine(_lib.ENGINE_TUNED)
    rng = np.random.default_rng([int(rpmax), int(pimax), len(kind)])
    A, B = _catalog(kind, 6000, rng, rpmax), _catalog(kind, 4000, rng, rpmax)
    e = np.linspace(0.5, rpmax, 6)
    binfile = bins_file(tmp_path, np.stack([e[:-1], e[1:]], 1))
    for cross in (False, True):
        kw = dict(autocorr=int(not cross), nthreads=4, binfile=binfile, RA1=A[0], DEC1=A[1], CZ1=A[2], pimax=pimax)
        if cross:
            kw.update(RA2=B[0], DEC2=B[1], CZ2=B[2])
        got = _abi.call_mocks(engine, "countpairs_mocks", options=opts(True), cosmology=1, **kw)
        want = _abi.call_mocks(oracle, "countpairs_mocks", "oracle_", options=opts(True), cosmology=1, **kw)
        assert_same("countpairs_mocks", got, want, "%s cross=%d" % (kind, cross))
        assert want["npairs"].sum() > 0
    os.environ["CORRFUNC_AMD_DENSE"] = "0"
