"""Gridding where many particles of a wave share a cell: few cells, sorted input, coincident points
and one crowded cell among many, single calls and batches, against the oracle."""
import numpy as np
import pytest

from corrfunc_amd import _abi, _lib
from helpers import assert_same, mode_kwargs, run, weights

pytestmark = pytest.mark.gpu

L = 60.0


def _points(kind, n, seed):
    rng = np.random.default_rng(seed)
    p = rng.uniform(0, L, (n, 3))
    if kind == "sorted":
        p = p[np.lexsort((p[:, 2] // 5, p[:, 1] // 5, p[:, 0] // 5))]
    elif kind == "coincident":
        p[n // 8:] = p[0]
    elif kind == "crowded":
        p[::2] = 21.0 + 0.5 * p[::2] / L
    elif kind == "pairs":      # two cells in turn, with a stranger now and then
        p[:] = np.where(np.arange(n)[:, None] % 2, 10.0, 50.0) + p / L
        p[::37] = rng.uniform(0, L, (len(p[::37]), 3))
    return [np.ascontiguousarray(p[:, d]) for d in range(3)]


@pytest.mark.parametrize("rmax", [4.0, 25.0])
@pytest.mark.parametrize("n", [1, 63, 65, 1999, 6001])
@pytest.mark.parametrize("kind", ["random", "sorted", "coincident", "crowded", "pairs"])
def test_shared_cells(engine, oracle, kind, n, rmax):
    _lib.set_engine(_lib.ENGINE_TUNED)
    X, W = _points(kind, n, n), weights(n, 1, np.float64)
    bins = np.linspace(0.0, rmax, 6)
    o = dict(periodic=True, boxsize=L, need_avg_sep=True)
    kw = mode_kwargs("countpairs", X, W, bins=bins, L=L)
    got = run(engine, "countpairs", options=_abi.make_options(**o), **kw)
    want = run(oracle, "countpairs", "oracle_", options=_abi.make_options(**o), **kw)
    assert_same("countpairs", got, want, what=kind)


def test_shared_cells_in_a_batch(engine, oracle):
    _lib.set_engine(_lib.ENGINE_TUNED)
    cats = [_points(k, n, 3) for k in ("pairs", "coincident", "sorted") for n in (65, 1999)]
    bins = np.linspace(0.0, 25.0, 6)
    o = dict(periodic=True, boxsize=L, need_avg_sep=True)
    for x, got in zip(cats, _lib.countpairs_batch([tuple(x) for x in cats], bins, options=_abi.make_options(**o))):
        want = run(oracle, "countpairs", "oracle_", options=_abi.make_options(**o),
                   **mode_kwargs("countpairs", x, bins=bins, L=L))
        assert np.array_equal(got["npairs"][1:], want["npairs"][1:])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [8191, 8192, 8193, 20479, 40000])
def test_few_crowded_cells(engine, oracle, n, dtype):
    """An open box of 8 cells, a thousand particles each and more (8192 is the line), as the second set
    of a cross-correlation; a last workgroup of any fill."""
    _lib.set_engine(_lib.ENGINE_TUNED)
    rng = np.random.default_rng(n)
    X, Y = [[rng.uniform(0, L, m).astype(dtype) for _ in range(3)] for m in (50, n)]
    bins = np.linspace(1.0, 1.5 * L, 6)
    o = dict(periodic=False, need_avg_sep=True, float_type=np.dtype(dtype).itemsize)
    kw = mode_kwargs("countpairs", X, weights(50, 1, dtype), Y, weights(n, 2, dtype), autocorr=0, bins=bins)
    got = run(engine, "countpairs", options=_abi.make_options(**o), **kw)
    assert _lib.last_stats()["nmesh"] == (2, 2, 2)
    want = run(oracle, "countpairs", "oracle_", options=_abi.make_options(**o), **kw)
    assert_same("countpairs", got, want)
