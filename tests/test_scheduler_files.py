"""Saved cost models say which features they were trained on; one of other features, or of a file that
does not say, is installed with a warning (results never depend on the model, the order of the work does)."""
import warnings

import numpy as np
import pytest

from corrfunc_amd import scheduler


@pytest.fixture
def installed(monkeypatch):
    """An installed model without the engine."""
    rng = np.random.default_rng(3)
    p, nm = rng.normal(size=scheduler.NPARAM).astype(np.float32), rng.normal(size=scheduler.NNORM).astype(np.float32)
    got = []
    monkeypatch.setattr(scheduler, "params", lambda: (p, nm))
    monkeypatch.setattr(scheduler, "set_params", lambda a, b: got.append((np.array(a), np.array(b))))
    return p, nm, got


def _installed(installed):
    p, nm, got = installed
    return len(got) == 1 and np.array_equal(got[0][0], p) and np.array_equal(got[0][1], nm)


def test_saved_and_loaded_in_silence(installed, tmp_path):
    f = str(tmp_path / "model.npz")
    scheduler.save(f)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        scheduler.load(f)
    assert _installed(installed)


@pytest.mark.parametrize("names", [None, ("log2(1+N1)", "dense", "z_overlap"), scheduler.FEATURE_NAMES[::-1]])
def test_model_of_other_features_warns(installed, tmp_path, names):
    f = str(tmp_path / "model.npz")
    extra = {} if names is None else {"features": np.array(names)}
    np.savez(f, params=installed[0], norm=installed[1], **extra)
    with pytest.warns(RuntimeWarning, match="train"):
        scheduler.load(f)
    assert _installed(installed)
