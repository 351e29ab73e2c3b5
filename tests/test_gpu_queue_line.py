"""The line from which the work queue hands out four items per atomic: 547,000 items, one a cell pair,
are above it with the 24 waves a CU that eight or fewer histogram copies leave (89 items a wave)."""
import numpy as np
import pytest

from corrfunc_amd import _abi, _lib
from helpers import assert_same, mode_kwargs, run, uniform

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,rmax,fetch", [("countpairs_rp_pi", 6.3, 4), ("countpairs_s_mu", 6.3, 4),
                                             ("countpairs", 6.3, 4), ("countpairs", 8.5, 1)])
def test_queue_batch_line(engine, oracle, monkeypatch, mode, rmax, fetch):
    monkeypatch.setenv("CORRFUNC_AMD_DENSE", "0")
    monkeypatch.delenv("CORRFUNC_AMD_FETCH", raising=False)
    _lib.set_engine(_lib.ENGINE_TUNED)
    n, L = (200000 if rmax < 7 else 100000), 100.0
    X = uniform(n, L, 17)
    kw = mode_kwargs(mode, X, bins=np.logspace(-0.5, np.log10(rmax), 11), L=L, pimax=rmax, nmu_bins=20)
    o = dict(periodic=True, boxsize=L, need_avg_sep=True)
    got = run(engine, mode, options=_abi.make_options(**o), **kw)
    st = _lib.last_stats()
    assert st["queue_fetch"] == fetch, st
    want = run(oracle, mode, "oracle_", options=_abi.make_options(**o), **kw)
    assert_same(mode, got, want)
