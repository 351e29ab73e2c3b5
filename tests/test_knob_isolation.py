"""An engine knob that one test leaves set does not reach the next."""
import os

import pytest


@pytest.mark.parametrize("again", [False, True])
def test_knob_of_another_test(again):
    assert "CORRFUNC_AMD_LEFT_BEHIND" not in os.environ
    os.environ["CORRFUNC_AMD_LEFT_BEHIND"] = "1"
