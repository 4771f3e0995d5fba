"""Segments and vector batches of the stochastic-volatility chain groups at their
edges: U and dU of the non-centred form where a thread's segment is around one
group of four steps and around the register limit of 16, and draws whose vectors
end inside, at and just past a batch of four elements per thread."""
import numpy as np
import pytest
import torch

from oracle import models as om

pytestmark = pytest.mark.gpu


def _data(T, C, seed):
    from numpyro_amd.workloads import make_sv
    rng = np.random.default_rng(seed)
    Z = rng.normal(size=(C, T + 2)).astype(np.float32)
    Z[:, 0] = np.log(rng.uniform(5, 15, C))
    Z[:, 1] = np.log(rng.uniform(0.02, 0.05, C))
    return make_sv(T, seed)[0], Z


def _engine(r, C, waves, **kw):
    from numpyro_amd.infer.hmc import Engine
    from numpyro_amd.models import StochasticVolatility
    eng = Engine(StochasticVolatility(r, noncentred=True), C, "NUTS", 0, **kw)
    eng.set_launch_shape(waves)
    return eng


@pytest.mark.parametrize("waves,T", [(1, 255), (1, 257), (1, 1024), (2, 513), (2, 2047), (4, 1023),
                                     (4, 1025), (4, 4096), (4, 4097), (8, 2049), (16, 3)])
def test_segment_edges(waves, T):
    from numpyro_amd import _lib
    C = 2
    r, Z = _data(T, C, T)
    eng = _engine(r, C, waves)
    z = torch.from_numpy(Z).cuda()
    pe = torch.empty(C, dtype=torch.float64, device="cuda")
    g = torch.empty((C, T + 2), dtype=torch.float32, device="cuda")
    _lib.check(_lib.load().nax_potential_grad(eng.h, _lib.ptr(z), T + 2, C, _lib.ptr(pe),
                                              _lib.ptr(g)))
    for c in range(C):  # bounds of the potential's oracle test
        u, gr = om.sv_nc_potential_grad(Z[c].astype(np.float64), np.asarray(r, np.float64))
        np.testing.assert_allclose(pe[c].item(), u, rtol=2e-6, atol=1e-3)
        np.testing.assert_allclose(g[c].cpu().numpy(), gr, rtol=2e-4,
                                   atol=2e-5 * (np.abs(gr).max() + 1))


@pytest.mark.parametrize("waves,T", [(1, 254), (1, 255), (2, 510), (4, 1021), (4, 1022), (4, 1023),
                                     (4, 60)])
def test_draws_at_batch_edges(waves, T):
    C, n = 2, 3
    r, Z = _data(T, C, T + 1)
    eng = _engine(r, C, waves, step_size=0.01, adapt_step_size=False, adapt_mass_matrix=False,
                  max_tree_depth=5)
    eng.init(torch.from_numpy(Z), np.arange(2 * C, dtype=np.uint32).reshape(C, 2))
    out = eng.run(n, collect_fields=("z", "potential_energy", "accept_prob"), size=n)
    z, pe = out["z"].cpu().numpy(), out["potential_energy"].cpu().numpy()
    for c in range(C):
        for i in range(n):  # a draw's energy is the potential at its position
            u, _ = om.sv_nc_potential_grad(z[c, i].astype(np.float64), np.asarray(r, np.float64))
            np.testing.assert_allclose(pe[c, i], u, rtol=2e-6, atol=1e-3)
    # a step of 0.01 is far below the stability limit: energy is conserved
    assert float(out["accept_prob"].min()) > 0.8
    assert np.abs(z[:, -1] - Z).max() > 0.0
