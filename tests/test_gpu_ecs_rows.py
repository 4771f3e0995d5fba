"""The subsampled evaluation's 16-row steps against float64: column chunks at
their edges (64, 65, 128, 192, 193, 256, 257, 512), subsamples around a step and
around a round of all waves, eight waves per chain (up to 256 chains) and four,
chain counts around the proxy kernel's four."""
import numpy as np
import pytest
import torch

from oracle import ecs

pytestmark = pytest.mark.gpu


def _case(N, D, m, C, degree, seed=0):
    from numpyro_amd.models import SubsampledLogisticRegression, potential_energy
    rng = np.random.default_rng(seed)
    X = rng.normal(size=(N, D)).astype(np.float32)
    beta = rng.normal(size=D) * 0.3
    y = (rng.uniform(size=N) < 1 / (1 + np.exp(-X @ beta))).astype(np.float32)
    ref = beta + 0.02
    mdl = SubsampledLogisticRegression(X, y, m, prior_scale=1.3, num_blocks=1, proxy_degree=degree,
                                       reference=ref if degree else None)
    idx = rng.integers(0, N, (C, m)).astype(np.int32)
    mdl.idx = torch.as_tensor(idx).cuda()
    mdl.keys = torch.zeros((C, 2), dtype=torch.int32, device="cuda")
    z = torch.tensor(beta + rng.normal(0, 0.05, (C, D)), dtype=torch.float32, device="cuda",
                     requires_grad=True)
    pe = potential_energy(mdl, z)
    (g,) = torch.autograd.grad(pe.sum(), z)
    st = ecs.taylor_stats(X, y, ref, degree) if degree else None
    return X, y, idx, st, z.detach().cpu().numpy().astype(np.float64), pe.detach().cpu(), g.cpu()


@pytest.mark.parametrize("degree", [0, 1, 2])
@pytest.mark.parametrize("D,m,C", [(1, 1, 1), (64, 16, 3), (65, 15, 4), (128, 17, 9), (192, 128, 5),
                                   (193, 129, 2), (256, 127, 257), (257, 65, 6), (512, 64, 300),
                                   (40, 65, 300), (130, 200, 256)])
def test_rows_vs_oracle(degree, D, m, C):
    N = 600
    X, y, idx, st, Z, pe, g = _case(N, D, m, C, degree)
    # fp32 logits and row sums against float64: as the potential's oracle test
    for c in sorted({0, 1, C // 2, C - 2, C - 1} & set(range(C))):
        u, gr = ecs.potential_grad(Z[c], idx[c], X, y, N, st, 1.3)
        np.testing.assert_allclose(pe[c].item(), u, rtol=2e-6)
        np.testing.assert_allclose(g[c].numpy(), gr, rtol=1e-4, atol=1e-4 * np.abs(gr).max())
