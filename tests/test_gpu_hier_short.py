"""One evaluation of short hierarchical regressions: models of up to 8 K rows take a
wave per chain, with the sums of a run at that launch shape; longer ones do not."""
import numpy as np
import pytest
import torch

from numpyro_amd import _lib
from numpyro_amd.models import HierarchicalLogistic

pytestmark = pytest.mark.gpu


def _eval(model, C, z, shape=None):
    from numpyro_amd.infer.hmc import Engine
    eng = Engine(model, C, "NUTS", 0)
    if shape is not None:
        eng.set_launch_shape(shape)
    pe = torch.zeros(C, dtype=torch.float64, device="cuda")
    g = torch.zeros((C, model.dim), device="cuda")
    torch.cuda.synchronize()
    _lib.check(_lib.load().nax_potential_grad(eng.h, _lib.ptr(z), model.dim, C, _lib.ptr(pe),
                                              _lib.ptr(g)), "potential_grad")
    return pe, g


@pytest.mark.parametrize("K", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("extra", [0, 1])
def test_short_models_take_a_wave_per_chain(K, extra):
    rng = np.random.default_rng(K)
    rows = [1, 8 * K + extra, 5 * K]
    Xs = [rng.normal(size=(n, 64)).astype(np.float32) for n in rows]
    ys = [(rng.uniform(size=n) < 0.4).astype(np.float32) for n in rows]
    model = HierarchicalLogistic(Xs, ys, chains_per_group=K)
    C = 3 * K
    z = torch.from_numpy((0.3 * rng.normal(size=(C, 66))).astype(np.float32)).cuda()
    pe, g = _eval(model, C, z)
    fpe, fg = _eval(model, C, z, shape=K)
    same = torch.equal(pe, fpe) and torch.equal(g, fg)
    assert same == (extra == 0)
    # sums of up to 129 residuals times |x| in another order, times tau = e^z
    torch.testing.assert_close(g, fg, rtol=0, atol=130 * 2.0 ** -24 * 130 * 4 * 3)
    torch.testing.assert_close(pe, fpe, rtol=1e-6, atol=1e-6)
