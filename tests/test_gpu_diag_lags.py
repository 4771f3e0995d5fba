"""The lag kernels of nax_diagnostics where their shape changes: parameters
around the tile widths (8, 16, 32), draws around the lag passes of 32 and the
lengths at which the tile narrows, chains fewer and more than the chain groups,
slow mixing (lags until the last), constant and non-finite draws, a slice of a
wider row; against the host formulas in float64.  Both sides sum in float64:
an autocovariance of S draws carries at most about S 2^-53 relative to the
variance, and at most S of them enter tau = n / ESS >= 1 / 2, so 1e-8 relative
holds with orders to spare for S <= 4096."""
import numpy as np
import pytest
import torch

from numpyro_amd import _lib
from numpyro_amd import diagnostics as nd

pytestmark = pytest.mark.gpu


def _chains(C, S, P, phi, seed):
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(C, S, P))
    for t in range(1, S):
        x[:, t] += phi * x[:, t - 1]
    return x.astype(np.float32)


def _check(x):
    ess, rhat = nd.device_diagnostics(torch.from_numpy(x))
    with np.errstate(all="ignore"):
        want = nd.effective_sample_size(x.astype(np.float64))
        want_r = nd.split_gelman_rubin(x.astype(np.float64))
    np.testing.assert_allclose(ess.cpu().numpy(), want, rtol=1e-8)
    if x.shape[1] >= 4:
        np.testing.assert_allclose(rhat.cpu().numpy(), want_r, rtol=1e-8)


@pytest.mark.parametrize("P", [1, 8, 9, 16, 17, 31, 32, 33, 70])
@pytest.mark.parametrize("S", [4, 31, 32, 33, 65, 97])
def test_tile_and_pass_edges(P, S):
    _check(_chains(3, S, P, 0.5, P * 100 + S))


@pytest.mark.parametrize("S", [608, 609, 1216, 1217, 2433])
def test_tile_width_rule(S):
    _check(_chains(2, S, 40, np.linspace(-0.5, 0.999, 40), S))


@pytest.mark.parametrize("C, P", [(1, 40), (2, 2500), (700, 40), (33, 600)])
def test_chain_groups_and_slow_mixing(C, P):
    _check(_chains(C, 300, P, np.linspace(0.0, 1.0, P), C + P))


def test_constant_and_non_finite_draws():
    x = _chains(4, 80, 36, 0.3, 5)
    x[:, :, 3] = 2.0
    x[1, 17, 5] = np.nan
    x[2, 40, 7] = np.inf
    ess, rhat = (t.cpu().numpy() for t in nd.device_diagnostics(torch.from_numpy(x)))
    bad = [3, 5, 7]
    assert np.isnan(ess[bad]).all() and np.isnan(rhat[bad]).all()
    keep = [i for i in range(36) if i not in bad]
    np.testing.assert_allclose(ess[keep], nd.effective_sample_size(x[:, :, keep]), rtol=1e-8)


def test_entry_point_without_a_workspace_and_refusals():
    lib = _lib.load()
    x = torch.from_numpy(_chains(3, 100, 20, 0.4, 9)).cuda()
    ess = torch.empty(20, dtype=torch.float64, device="cuda")
    want, _ = nd.device_diagnostics(x)
    _lib.check(lib.nax_diagnostics(_lib.ptr(x), 3, 100, 20, _lib.ptr(ess), None), "diagnostics")
    assert torch.equal(ess, want)
    assert lib.nax_diagnostics_workspace(3, 4097, 20) == 0
    assert lib.nax_diagnostics_ws(_lib.ptr(x), 3, 100, 20, _lib.ptr(ess), None, _lib.ptr(ess),
                                  8) == -22
