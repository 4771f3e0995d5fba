"""Small residuals in the matrix-core kernel's X^T R (logit_split_kernel): rare
events on one-hot and binary columns, where thousands of rows share one residual
far below 1 and an error of it has the same sign in all of them.

Reference: float64.  Bound of a gradient entry, relative to the sum of its |r x|: a
logit of K terms that are not zero carries K + 1 roundings, each at most 2^-24
of sum |x z| =: M; the exponential's argument a = |l| log2 e carries 1.5 roundings
2^-24 a, scaled by ln 2, and exp2, 1 + e, reciprocal and product together 6 of 2^-24;
the sums over a row split take 5 roundings per 32 rows (two products of R's grid
terms with each half tile, and the tile's fine terms), each at most 2^-24 of what
the split holds.  A split has at most 512 of the 131,072 rows."""
import math

import pytest
import torch

from numpyro_amd import _lib

pytestmark = pytest.mark.gpu

N = 131072


def _rare(D, rate, C, seed):
    """Eight one-hot columns at the given event rate, then binary columns that
    no chain uses; K = 1 term of a logit is not zero."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    X = (torch.rand((N, D), generator=g, device="cuda") < 0.1).float()
    X[:, :8] = torch.nn.functional.one_hot(
        torch.randint(0, 8, (N,), generator=g, device="cuda"), 8).float()
    z = torch.zeros((C, D), device="cuda")
    z[:, :8] = math.log(rate / (1 - rate)) + 0.3 * torch.randn((C, 8), generator=g, device="cuda")
    y = (torch.rand(N, generator=g, device="cuda") < rate).float()
    return X, y, z


def _grad(X, y, z, x_dtype, kernel):
    from numpyro_amd.infer.hmc import Engine
    from numpyro_amd.models import LogisticRegression
    C, D = z.shape
    eng = Engine(LogisticRegression(X, y, x_dtype=x_dtype, kernel=kernel), C, "NUTS", 0)
    pe = torch.full((C,), float("nan"), dtype=torch.float64, device="cuda")
    g = torch.full((C, D), float("nan"), device="cuda")
    torch.cuda.synchronize()
    _lib.check(_lib.load().nax_potential_grad(eng.h, _lib.ptr(z), D, C, _lib.ptr(pe),
                                              _lib.ptr(g)), "potential_grad")
    return g.double()


@pytest.mark.parametrize("x_dtype, C", [("fp32", 130), ("fp8", 33)])
@pytest.mark.parametrize("D, rate", [(8, 1e-2), (8, 1e-3), (8, 1e-4), (40, 1e-3), (90, 1e-4),
                                     (128, 1e-3), (161, 1e-2), (256, 1e-3), (256, 1e-4)])
def test_rare_events_keep_their_bits(D, rate, x_dtype, C):
    X, y, z = _rare(D, rate, C, D)  # 0 and 1 are exact in every storage form
    got = _grad(X, y, z, x_dtype, "auto")
    x, z64 = X.double(), z.double()
    l = x @ z64.T
    r = torch.sigmoid(l) - y.double()[:, None]
    want = r.T.contiguous() @ x + z64
    M = float(l.abs().max())
    steps = 5 * 512 / 32
    eps = (2 * M + 1.5 * math.log(2) * 1.4427 * M + 6 + steps) * 2.0 ** -24
    bound = eps * (r.abs().T.contiguous() @ x.abs()) + 2.0 ** -23 * z64.abs() + 1e-9
    assert ((got - want).abs() <= bound).all(), float(((got - want).abs() / bound).max())
