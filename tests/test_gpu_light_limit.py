"""The line between the light kernel (one lane per cell pair) and the persistent kernel's work list:
the limit of 128 tests a cell pair, and sparse catalogs through either kernel, against the oracle."""
import numpy as np
import pytest

from corrfunc_amd import _abi, _lib, scheduler
from helpers import MODES, assert_same, mode_kwargs, run, weights

pytestmark = pytest.mark.gpu

L = 150.0
BINS = np.logspace(-1, np.log10(6.0), 9)


@pytest.fixture(autouse=True)
def _tuned(engine, monkeypatch):
    monkeypatch.setenv("CORRFUNC_AMD_DENSE", "0")
    monkeypatch.delenv("CORRFUNC_AMD_LIGHT", raising=False)
    _lib.set_engine(_lib.ENGINE_TUNED)
    scheduler.set_scheduler("none")  # one item per 64 primaries: no slices of heavy cell pairs
    yield
    scheduler.set_scheduler("learned")


def _sparse(clump, seed):
    """A thin background and `clump` points in one cell (39-42, 39-42, 36-42) that has no others."""
    rng = np.random.default_rng(seed)
    p = rng.uniform(0, L, (9000, 3))
    p = p[np.any((p < 38.9) | (p > 42.1), axis=1)]
    p = np.concatenate([p, rng.uniform(39.3, 41.7, (clump, 3)), [[0.0] * 3, [L] * 3]])
    return [np.ascontiguousarray(p[:, d]) for d in range(3)]


def _compare(engine, oracle, mode, X, avg):
    W = weights(len(X[0]), 3, np.float64) if avg else None
    o = dict(periodic=True, boxsize=L, need_avg_sep=avg)
    kw = mode_kwargs(mode, X, W, bins=BINS, L=L, pimax=6.0, nmu_bins=5)
    got = run(engine, mode, options=_abi.make_options(**o), **kw)
    st = _lib.last_stats()
    want = run(oracle, mode, "oracle_", options=_abi.make_options(**o), **kw)
    assert_same(mode, got, want)
    return st


@pytest.mark.parametrize("clump,listed", [(2, 0), (11, 0), (12, 1), (33, 1), (64, 1)])
def test_limit_of_a_lane(engine, oracle, clump, listed):
    """One cell pair (the clump's cell with itself, clump^2 tests) crosses the limit: its chunks of 64
    primaries are the work list. No lane takes a long chain, however few tests the average has."""
    st = _compare(engine, oracle, "countpairs", _sparse(clump, clump), True)
    assert st["num_work_items"] == listed, st


@pytest.mark.parametrize("limit", ["0", "1", "1024"])
@pytest.mark.parametrize("avg", [False, True])
@pytest.mark.parametrize("mode", MODES)
def test_either_kernel(engine, oracle, monkeypatch, mode, avg, limit):
    monkeypatch.setenv("CORRFUNC_AMD_LIGHT", limit)
    st = _compare(engine, oracle, mode, _sparse(31, 5), avg)
    assert (st["num_work_items"] >= st["num_cell_pairs"]) == (limit == "0"), st
    assert (st["num_work_items"] == 0) == (limit == "1024"), st
