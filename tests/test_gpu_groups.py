"""Cells of every size the grouped pair kernel distinguishes, against the oracle: one group of 16
secondaries and less, chunk edges (64), windows that are box-tested and not, the largest cell one
wave sorts (512) and the next, more than 64 groups. A dense ball inside one cell gives the size, a
thin uniform background the neighbours; counts are equal, averages within the summation-order
bound used throughout (1e-10)."""
import os

import numpy as np
import pytest

from corrfunc_amd import _abi, _lib
from helpers import MODES, assert_same, mode_kwargs, run, weights

pytestmark = pytest.mark.gpu

L = 120.0
BINS = np.concatenate([[0.0], np.logspace(-1.5, np.log10(14.0), 12)])


def _ball(n, dtype, seed, sigma=0.8, nback=700):
    rng = np.random.default_rng(seed)
    p = np.concatenate([rng.normal(31.0, sigma, (n, 3)), rng.uniform(0, L, (nback, 3))]).astype(dtype)
    p = p[rng.permutation(len(p))]
    return [np.ascontiguousarray(p[:, d]) for d in range(3)]


@pytest.mark.parametrize("isa", ["fallback", "avx512f"])
@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n", [1, 15, 17, 33, 64, 65, 500, 530, 1100, 2600])
def test_cell_sizes(engine, oracle, n, mode, isa):
    os.environ["CORRFUNC_AMD_DENSE"] = "0"
    _lib.set_engine(_lib.ENGINE_TUNED)
    dtype = np.float32 if n % 2 else np.float64
    X = _ball(n, dtype, n)
    W = weights(len(X[0]), n + 1, dtype)
    kw = mode_kwargs(mode, X, W, bins=BINS, L=L, pimax=20.0, nmu_bins=7)
    for avg in (True, False):
        o = dict(periodic=True, boxsize=L, need_avg_sep=avg, isa=isa, float_type=np.dtype(dtype).itemsize)
        if not avg:
            kw.pop("weights1", None)
            kw.pop("weight_type", None)
        got = run(engine, mode, options=_abi.make_options(**o), **kw)
        want = run(oracle, mode, "oracle_", options=_abi.make_options(**o), **kw)
        assert_same(mode, got, want, what="ball of %d" % n)


@pytest.mark.parametrize("mode", MODES[:3])
def test_cross_of_unequal_cells(engine, oracle, mode):
    os.environ["CORRFUNC_AMD_DENSE"] = "0"
    _lib.set_engine(_lib.ENGINE_TUNED)
    X, Y = _ball(70, np.float64, 5), _ball(1500, np.float64, 6, sigma=4.0)
    WX, WY = weights(len(X[0]), 7, np.float64), weights(len(Y[0]), 8, np.float64)
    for periodic in (True, False):
        o = dict(periodic=periodic, boxsize=L if periodic else None, need_avg_sep=True)
        for a, wa, b, wb in ((X, WX, Y, WY), (Y, WY, X, WX)):
            kw = mode_kwargs(mode, a, wa, b, wb, autocorr=0, bins=BINS, L=L, pimax=20.0, nmu_bins=7)
            got = run(engine, mode, options=_abi.make_options(**o), **kw)
            want = run(oracle, mode, "oracle_", options=_abi.make_options(**o), **kw)
            assert_same(mode, got, want, what="cross")


def test_nan_coordinates_count_in_no_pair(engine):
    """A particle with a NaN coordinate is in no pair with another one, whichever group it lands in
    (with rmin = 0 every particle, this one too, counts itself in the first bin)."""
    os.environ["CORRFUNC_AMD_DENSE"] = "0"
    _lib.set_engine(_lib.ENGINE_TUNED)
    X = _ball(900, np.float64, 11, sigma=3.0)
    o = dict(periodic=True, boxsize=L, need_avg_sep=True)
    ref = run(engine, "countpairs", options=_abi.make_options(**o), **mode_kwargs("countpairs", X, bins=BINS, L=L))
    for d in range(3):
        Y = [np.concatenate([c, [31.0 if k != d else np.nan]]) for k, c in enumerate(X)]
        got = run(engine, "countpairs", options=_abi.make_options(**o), **mode_kwargs("countpairs", Y, bins=BINS, L=L))
        assert got["npairs"][1] == ref["npairs"][1] + 1
        assert np.array_equal(got["npairs"][2:], ref["npairs"][2:])
        assert np.allclose(got["ravg"][2:], ref["ravg"][2:], rtol=1e-10, atol=0)
