"""Sparse scans over cells of just under, at and over 64 and 128 groups of secondaries (1024 and 2048):
queue entries count from the first of 64 groups, so survivors that wait at the end of one such batch
are decided before the next starts. No dense groups, one and two survivors per lane and drain,
against the oracle."""
import numpy as np
import pytest

from corrfunc_amd import _abi, _lib
from helpers import assert_same, mode_kwargs, run, weights

pytestmark = pytest.mark.gpu

L = 120.0
BINS = np.logspace(-1, np.log10(14.0), 9)


def _one_cell(n, nback, seed):
    """n points in the cell (30-37.5, 30-37.5, 30-45) and nback all over the box."""
    rng = np.random.default_rng(seed)
    p = np.concatenate([rng.uniform([30.2, 30.2, 31.0], [34.8, 34.8, 44.0], (n, 3)), rng.uniform(0, L, (nback, 3)),
                        [[0.0] * 3, [L] * 3]])
    p = p[rng.permutation(len(p))]
    return [np.ascontiguousarray(p[:, d]) for d in range(3)]


@pytest.fixture(autouse=True)
def _sparse(engine, monkeypatch):
    monkeypatch.setenv("CORRFUNC_AMD_DENSE", "2")
    _lib.set_engine(_lib.ENGINE_TUNED)


def _compare(engine, oracle, mode, X, Y=None):
    W = weights(len(X[0]), 1, np.float64)
    W2 = weights(len(Y[0]), 2, np.float64) if Y is not None else None
    o = dict(periodic=True, boxsize=L, need_avg_sep=True)
    kw = mode_kwargs(mode, X, W, Y, W2, autocorr=int(Y is None), bins=BINS, L=L, pimax=14.0, nmu_bins=5)
    got = run(engine, mode, options=_abi.make_options(**o), **kw)
    want = run(oracle, mode, "oracle_", options=_abi.make_options(**o), **kw)
    assert_same(mode, got, want)


@pytest.mark.parametrize("drain", ["1", "2"])
@pytest.mark.parametrize("mode", ["countpairs", "countpairs_rp_pi", "countpairs_s_mu"])
@pytest.mark.parametrize("n", [1008, 1023, 1024, 1025, 1041, 2047, 2048, 2049, 3100])
def test_cells_around_64_groups(engine, oracle, monkeypatch, mode, n, drain):
    monkeypatch.setenv("CORRFUNC_AMD_DRAIN_PAIRS", drain)
    _compare(engine, oracle, mode, _one_cell(n, 0, n))
    _compare(engine, oracle, mode, _one_cell(67, 300, n + 1), _one_cell(n, 0, n))
