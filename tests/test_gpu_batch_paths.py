"""A batch gridded jointly and catalog by catalog (the way of the largest ones): the same cell pairs and
the same results, equal to the oracle's."""
import numpy as np
import pytest

from corrfunc_amd import _abi, _lib
from helpers import mode_kwargs, run, weights

pytestmark = pytest.mark.gpu

L = 150.0


def _catalog(n, clump, dtype, seed):
    rng = np.random.default_rng(seed)
    p = np.concatenate([rng.uniform(0, L, (n, 3)), rng.normal(40.0, 0.4, (clump, 3))]).astype(dtype)
    return [np.ascontiguousarray(p[:, d]) for d in range(3)]


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("rmax", [6.0, 40.0])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_joint_and_single_gridding(engine, oracle, monkeypatch, dtype, rmax, weighted):
    _lib.set_engine(_lib.ENGINE_TUNED)
    sizes = [(0, 0), (1, 0), (3000, 700), (0, 0), (2, 0), (6000, 17), (500, 2000), (0, 0)]
    cats = [_catalog(n, c, dtype, 7 * k) for k, (n, c) in enumerate(sizes)]
    W = [weights(len(x[0]), k, dtype) for k, x in enumerate(cats)] if weighted else None
    bins = np.logspace(-1, np.log10(rmax), 9)
    o = dict(periodic=True, boxsize=L, need_avg_sep=True, float_type=np.dtype(dtype).itemsize)
    stats = []
    for limit in (None, "0"):
        monkeypatch.delenv("CORRFUNC_AMD_BATCH_CAND", raising=False)
        if limit is not None:
            monkeypatch.setenv("CORRFUNC_AMD_BATCH_CAND", limit)
        res = _lib.countpairs_batch([tuple(x) for x in cats], bins, options=_abi.make_options(**o), weights=W)
        stats.append(_lib.last_stats())
        for k, (x, got) in enumerate(zip(cats, res)):
            want = run(oracle, "countpairs", "oracle_", options=_abi.make_options(**o),
                       **mode_kwargs("countpairs", x, W[k] if weighted else None, bins=bins, L=L))
            assert np.array_equal(got["npairs"][1:], want["npairs"][1:]), (limit, k)
            for key in ("ravg", "weightavg"):
                assert np.allclose(got[key][1:], want[key][1:], rtol=1e-10, atol=0), (limit, k, key)
    for key in ("num_cell_pairs", "tested_pairs"):
        assert stats[0][key] == stats[1][key], key
