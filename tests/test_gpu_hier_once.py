"""The one-shot evaluation of ragged hierarchical regressions against the float64
oracle at the edges of its tiles: 32 rows per wave and 8 waves, LDS rows padded
when D is a multiple of 8, 16-byte reads when D is a multiple of 4, chains in
groups of 4, and models split over blocks."""
import numpy as np
import pytest
import torch

from numpyro_amd.models import HierarchicalLogistic, potential_energy
from oracle import models as om

pytestmark = pytest.mark.gpu

SHAPES = [(1, 64), (31, 1), (32, 2), (33, 3), (255, 8), (256, 12), (257, 30), (288, 31),
          (4999, 56), (5000, 63), (3001, 48), (40, 5)]


@pytest.mark.parametrize("K", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("transform", ["exp", "softplus"])
def test_one_shot_against_oracle(K, transform):
    rng = np.random.default_rng(K)
    Xs = [rng.normal(size=s).astype(np.float32) for s in SHAPES]
    ys = [(rng.uniform(size=n) < 0.4).astype(np.float32) for n, _ in SHAPES]
    m = HierarchicalLogistic(Xs, ys, chains_per_group=K, positive_transform=transform)
    Z = np.zeros((len(SHAPES) * K, m.dim), np.float32)
    for c in range(len(Z)):
        d = SHAPES[c // K][1]
        Z[c, :d + 2] = 0.3 * rng.normal(size=d + 2)
    z = torch.from_numpy(Z).cuda().requires_grad_()
    U = potential_energy(m, z)
    U.sum().backward()
    for c in range(len(Z)):
        n, d = SHAPES[c // K]
        zc = Z[c, :d + 2].astype(np.float64)
        X, y = Xs[c // K], ys[c // K]
        f = lambda v: om.hier_potential(v, X, y, positive=transform)
        # a logit is a sum of d rounded products in four chains: |error| <=
        # (d / 4 + 4) 2^-24 sum |x b|; U's terms are 1-Lipschitz in it
        b = zc[d] + (np.exp(zc[d + 1]) if transform == "exp" else np.log1p(np.exp(zc[d + 1]))) * zc[:d]
        lim = (d / 4 + 8) * 2.0 ** -24 * (np.abs(X) @ np.abs(b) + 1.0)
        assert abs(U[c].item() - f(zc)) <= lim.sum() + 1e-6
        # residuals are 1/4-Lipschitz in the logit; n terms of |x| <= max |x| are added in
        # fp32, and eta, tau multiply the column sums
        if transform == "exp":
            g = om.hier_potential_grad(zc, X, y)[1]
        else:
            g = om.central_fd(f, zc)
        col = np.abs(X).T @ (lim + 2.0 ** -22) + n / 64 * 2.0 ** -24 * np.abs(X).sum(0)
        amp = (1 + np.exp(abs(zc[d + 1]))) * (1 + np.abs(zc[:d]).max())
        fd = 1e-5 * (1 + abs(f(zc))) if transform != "exp" else 0.0
        assert np.abs(z.grad[c, :d + 2].cpu().numpy() - g).max() <= amp * col.sum() + 1e-5 + fd
    # a chain with an infinite latent has no bearing on its neighbours
    if K > 1:
        Z2 = Z.copy()
        Z2[0, 0] = np.inf
        U2 = potential_energy(m, torch.from_numpy(Z2).cuda())
        assert torch.equal(U2[1:], U.detach()[1:])
