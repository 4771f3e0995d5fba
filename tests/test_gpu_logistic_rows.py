"""The row-tile kernel of the logistic potential (fp32, up to 31 chains) against
float64: edges of its 32-row tiles and 64-column blocks, 16-byte and single
reads, LDS rows with and without padding, several tiles per wave, 1 to 31
chains, and a design that starts off a 16-byte boundary."""
import numpy as np
import pytest
import torch

from numpyro_amd.models import LogisticRegression, potential_energy

pytestmark = pytest.mark.gpu

# (n, d, chains); d <= 64 with few chains and few rows takes another kernel
CASES = [(1, 1, 17), (31, 4, 31), (33, 63, 20), (32, 64, 17), (129, 65, 1), (1, 256, 3),
         (1000, 128, 4), (5000, 129, 5), (300, 192, 8), (4097, 255, 9), (35000, 256, 16),
         (140001, 8, 2), (270000, 5, 1), (20011, 200, 31)]


def _eval(X, y, z):
    z = z.clone().requires_grad_()
    U = potential_energy(LogisticRegression(X, y), z)
    U.sum().backward()
    return U.detach(), z.grad


@pytest.mark.parametrize("n, d, C", CASES)
def test_rows_against_float64(n, d, C):
    g = torch.Generator().manual_seed(n + d + C)
    buf = torch.randn(n * d + 1, generator=g)
    X = buf[1:].view(n, d)
    y = (torch.rand(n, generator=g) < 0.4).float()
    z = torch.randn(C, d, generator=g) / d ** 0.5
    U, gr = _eval(X.cuda(), y.cuda(), z.cuda())
    Xd, zd, yd = X.double(), z.double(), y.double()
    l = Xd @ zd.T
    want = (torch.nn.functional.softplus(l) - yd[:, None] * l).sum(0) + (
        0.5 * zd ** 2 + 0.5 * np.log(2 * np.pi)).sum(1)
    r = torch.sigmoid(l) - yd[:, None]
    wg = r.T @ Xd + zd
    # a logit is d rounded multiply-adds, the terms a few roundings of 1 + |l|
    lim = d * 2.0 ** -24 * (Xd.abs() @ zd.abs().T) + 2.0 ** -21 * (1 + l.abs())
    assert ((U.cpu() - want).abs() <= lim.sum(0) + 1e-9 * want.abs()).all()
    # residuals are 1/4-Lipschitz in the logit; a column's products pass through at most
    # 200 sums: rows of a tile, tiles of a wave, waves, row splits of a group
    gl = (lim / 4 + 2.0 ** -22).T @ Xd.abs() + 200 * 2.0 ** -24 * (r.abs().T @ Xd.abs() + zd.abs())
    assert ((gr.cpu() - wg).abs() <= gl).all()
    # off a 16-byte boundary: the same numbers
    base = torch.empty(n * d + 1, device="cuda")
    Xo = base[1:].view(n, d)
    Xo.copy_(X)
    U2, g2 = _eval(Xo, y.cuda(), z.cuda())
    assert torch.equal(U, U2) and torch.equal(gr, g2)
    if C > 1:  # a chain at infinity has no bearing on the others
        zi = z.clone()
        zi[0, 0] = float("inf")
        U3, g3 = _eval(X.cuda(), y.cuda(), zi.cuda())
        assert torch.equal(U[1:], U3[1:]) and torch.equal(gr[1:], g3[1:])
