"""Diagnostics of up to 256 draws, whose lags are all taken in one round where their
workgroups fit the chip: draws around the passes of 32 lags and the limit, slow
mixing (every lag counts), several tiles and groups, both sides of the rule."""
import pytest

from test_gpu_diag_lags import _chains, _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [2, 3, 34, 63, 66, 255, 256, 257])
@pytest.mark.parametrize("C, P, phi", [(1, 1, 0.99), (4, 70, 0.9), (300, 33, 0.995), (2, 1500, 0.5),
                                       (64, 8, 0.999)])
def test_short_chains(S, C, P, phi):
    _check(_chains(C, S, P, phi, S + P))
