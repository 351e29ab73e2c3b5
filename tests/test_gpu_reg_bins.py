"""1-D counts of groups that span few bins, kept in registers, where their bins end at rmax."""
import numpy as np
import pytest

from corrfunc_amd import _abi, _lib
from helpers import assert_same, mode_kwargs, run

pytestmark = pytest.mark.gpu

MODES_1D = ("countpairs", "countpairs_xi", "countpairs_wp")


def _lattice(n, drop, dtype):
    """Unit lattice of n^3 points less the last `drop`, whose last cell ends in a partial chunk."""
    g = np.arange(n, dtype=np.float64) + 0.5
    p = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    p = p[:len(p) - drop].astype(dtype)
    return [np.ascontiguousarray(p[:, d]) for d in range(3)]


@pytest.fixture(autouse=True)
def _tuned(engine, monkeypatch):
    monkeypatch.setenv("CORRFUNC_AMD_DENSE", "0")
    _lib.set_engine(_lib.ENGINE_TUNED)


@pytest.mark.parametrize("drop", [0, 1, 63, 117])
@pytest.mark.parametrize("mode", MODES_1D)
def test_lattice_separations_just_below_rmax(engine, oracle, mode, drop):
    """Separations of 10 with rmax a few ulps above: every chunk has pairs that replay the pruning
    rules, among them the partial ones (250 particles a cell), whose idle lanes have none."""
    dtype = np.float32 if drop % 2 else np.float64
    X = _lattice(30, drop, dtype)
    bins = np.array([0.5, 5.0, 10.0 * (1 + 2e-10)])
    o = dict(periodic=True, boxsize=30.0, need_avg_sep=False, isa="avx512f", float_type=np.dtype(dtype).itemsize)
    kw = mode_kwargs(mode, X, bins=bins, L=30.0, pimax=12.0)
    got = run(engine, mode, options=_abi.make_options(**o), **kw)
    want = run(oracle, mode, "oracle_", options=_abi.make_options(**o), **kw)
    assert_same(mode, got, want, what="lattice")
    assert want["npairs"][-1] > 0


def test_lattice_in_a_captured_batch(engine, oracle):
    """The same in a graph, whose record arrays end right behind the last particle."""
    cats = [_lattice(30, d, np.float64) for d in (0, 63)]
    dev = [[_lib.DeviceArray(a) for a in x] for x in cats]
    bins = np.array([0.5, 5.0, 10.0 * (1 + 2e-10)])
    o = dict(periodic=True, boxsize=30.0, need_avg_sep=False)
    g = _lib.BatchGraph([tuple(d) for d in dev], bins, options=_abi.make_options(**o))
    try:
        for _ in range(3):
            for x, got in zip(cats, g.launch()):
                want = run(oracle, "countpairs", "oracle_", options=_abi.make_options(**o),
                           **mode_kwargs("countpairs", x, bins=bins, L=30.0))
                assert_same("countpairs", got, want, what="graph")
    finally:
        g.close()


def _edge_file(tmp_path, pairs):
    f = tmp_path / "bins"
    f.write_text("".join("%r %r\n" % p for p in pairs))
    return str(f)


@pytest.mark.parametrize("upper", [(5.0, 12.0, 9.0), (2.0, 12.0, 30.0, 9.0), (9.0, 9.0), (10.0, 9.0), (3.0, 6.0, 9.0)])
@pytest.mark.parametrize("mode", MODES_1D)
def test_last_edge_below_an_earlier_one(engine, oracle, tmp_path, mode, upper):
    """rmax is the last line's upper edge, whichever edges lie above it: counts end there."""
    rng = np.random.default_rng(len(upper))
    X = [rng.uniform(0, 40.0, 40000) for _ in range(3)]
    lower = (1.0,) + upper[:-1]
    o = dict(periodic=True, boxsize=40.0, need_avg_sep=False)
    kw = mode_kwargs(mode, X, bins=_edge_file(tmp_path, list(zip(lower, upper))), L=40.0, pimax=12.0)
    got = run(engine, mode, options=_abi.make_options(**o), **kw)
    want = run(oracle, mode, "oracle_", options=_abi.make_options(**o), **kw)
    assert_same(mode, got, want, what="edges %s" % (upper,))


def test_last_edge_below_an_earlier_one_in_a_captured_batch(engine, oracle, tmp_path):
    rng = np.random.default_rng(9)
    cats = [[rng.uniform(0, 40.0, 40000) for _ in range(3)] for _ in range(2)]
    dev = [[_lib.DeviceArray(a) for a in x] for x in cats]
    bins = _edge_file(tmp_path, [(1.0, 5.0), (5.0, 12.0), (12.0, 9.0)])
    o = dict(periodic=True, boxsize=40.0, need_avg_sep=False)
    g = _lib.BatchGraph([tuple(d) for d in dev], bins, options=_abi.make_options(**o))
    try:
        for x, got in zip(cats, g.launch()):
            want = run(oracle, "countpairs", "oracle_", options=_abi.make_options(**o),
                       **mode_kwargs("countpairs", x, bins=bins, L=40.0))
            assert_same("countpairs", got, want, what="graph")
    finally:
        g.close()
