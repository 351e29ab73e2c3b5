"""Sparse grids, whose light cell pairs (at most 1024 tests) are counted one lane per cell pair and
whose heavy ones by the persistent kernel: all modes against the oracle, with a clump that makes a
few cell pairs heavy, at sizes around the limit, and batches with empty and one-point catalogs."""
import os

import numpy as np
import pytest

from corrfunc_amd import _abi, _lib
from helpers import MODES, assert_same, mode_kwargs, run, weights

pytestmark = pytest.mark.gpu

L = 150.0
BINS = np.logspace(-1, np.log10(6.0), 9)


def _sparse(n, clump, dtype, seed):
    rng = np.random.default_rng(seed)
    p = np.concatenate([rng.uniform(0, L, (n, 3)), rng.normal(40.0, 0.4, (clump, 3))]).astype(dtype)
    return [np.ascontiguousarray(p[:, d]) for d in range(3)]


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("clump", [0, 15, 16, 17, 31, 32, 33, 46, 200])
@pytest.mark.parametrize("avg", [False, True])
def test_light_cell_pairs(engine, oracle, mode, clump, avg):
    os.environ["CORRFUNC_AMD_DENSE"] = "0"
    _lib.set_engine(_lib.ENGINE_TUNED)
    dtype = np.float32 if clump % 2 else np.float64
    X = _sparse(9000, clump, dtype, clump)
    W = weights(len(X[0]), 3, dtype) if avg else None
    o = dict(periodic=True, boxsize=L, need_avg_sep=avg, float_type=np.dtype(dtype).itemsize)
    kw = mode_kwargs(mode, X, W, bins=BINS, L=L, pimax=8.0, nmu_bins=5)
    got = run(engine, mode, options=_abi.make_options(**o), **kw)
    want = run(oracle, mode, "oracle_", options=_abi.make_options(**o), **kw)
    assert_same(mode, got, want, what="clump of %d" % clump)


def test_light_cross_open_box(engine, oracle):
    os.environ["CORRFUNC_AMD_DENSE"] = "0"
    _lib.set_engine(_lib.ENGINE_TUNED)
    X, Y = _sparse(4000, 30, np.float64, 1), _sparse(9000, 60, np.float64, 2)
    for mode in MODES[:3]:
        o = dict(periodic=False, need_avg_sep=True)
        kw = mode_kwargs(mode, X, weights(len(X[0]), 4, np.float64), Y, weights(len(Y[0]), 5, np.float64), autocorr=0,
                         bins=BINS, L=L, pimax=8.0, nmu_bins=5)
        got = run(engine, mode, options=_abi.make_options(**o), **kw)
        want = run(oracle, mode, "oracle_", options=_abi.make_options(**o), **kw)
        assert_same(mode, got, want, what="cross")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_batch_of_unequal_catalogs(engine, oracle, dtype):
    os.environ["CORRFUNC_AMD_DENSE"] = "0"
    _lib.set_engine(_lib.ENGINE_TUNED)
    sizes = [(0, 0), (1, 0), (3000, 700), (0, 0), (2, 0), (9000, 17), (500, 2000), (0, 0)]
    cats = [_sparse(n, c, dtype, 7 * k) for k, (n, c) in enumerate(sizes)]
    W = [weights(len(x[0]), k, dtype) for k, x in enumerate(cats)]
    o = dict(periodic=True, boxsize=L, need_avg_sep=True, float_type=np.dtype(dtype).itemsize)
    res = _lib.countpairs_batch([tuple(x) for x in cats], BINS, options=_abi.make_options(**o), weights=W)
    for x, w, got in zip(cats, W, res):
        want = run(oracle, "countpairs", "oracle_", options=_abi.make_options(**o),
                   **mode_kwargs("countpairs", x, w, bins=BINS, L=L))
        assert np.array_equal(got["npairs"][1:], want["npairs"][1:])
        for k in ("ravg", "weightavg"):
            assert np.allclose(got[k][1:], want[k][1:], rtol=1e-10, atol=0)


def test_graph_of_sparse_catalogs(engine, oracle):
    """A captured batch has no light kernel: its work list takes every cell pair."""
    os.environ["CORRFUNC_AMD_DENSE"] = "0"
    _lib.set_engine(_lib.ENGINE_TUNED)
    cats = [_sparse(9000, c, np.float64, 50 + c) for c in (0, 40, 0)]
    dev = [[_lib.DeviceArray(a) for a in x] for x in cats]
    o = dict(periodic=True, boxsize=L, need_avg_sep=True)
    g = _lib.BatchGraph([tuple(d) for d in dev], BINS, options=_abi.make_options(**o))
    try:
        for _ in range(2):
            for x, got in zip(cats, g.launch()):
                want = run(oracle, "countpairs", "oracle_", options=_abi.make_options(**o),
                           **mode_kwargs("countpairs", x, bins=BINS, L=L))
                assert_same("countpairs", got, want, what="graph")
    finally:
        g.close()


@pytest.mark.parametrize("rmax", [1.45, 2.6, 30.0])
def test_scans_of_every_depth(engine, oracle, rmax):
    """27 million candidate cell pairs (a scan of scanned block sums), 4 million, and a few hundred
    (one block)."""
    os.environ["CORRFUNC_AMD_DENSE"] = "0"
    _lib.set_engine(_lib.ENGINE_TUNED)
    X = _sparse(20000, 300, np.float64, 77)
    bins = np.linspace(0.1, rmax, 5)
    o = dict(periodic=True, boxsize=L, need_avg_sep=True)
    kw = mode_kwargs("countpairs", X, bins=bins, L=L)
    got = run(engine, "countpairs", options=_abi.make_options(**o), **kw)
    want = run(oracle, "countpairs", "oracle_", options=_abi.make_options(**o), **kw)
    assert_same("countpairs", got, want, what="rmax %g" % rmax)
