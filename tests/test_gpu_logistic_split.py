"""The matrix-core kernel for fp32 and fp8 designs (logit_split_kernel) at the
edges of its tiles and rules: columns around the multiples of 8 and 32, rows
around the tile of 32 and the split's lower limit, chains around the wave (32)
and block (128), the two-term split, the fp32 form it falls back to and fp8
codes, positions with infinities or NaN, and the compacted list of chains of a
sampling run.

Reference: float64 on the design the form stands for.  Bound of a gradient
entry: the logit carries at most (D + 1) 2^-24 of sum |x z| (a chain of fused
multiply-adds) and moves r by a quarter of that, r itself 2^-21 (hardware exp and
reciprocal, and the two terms), each term of X^T R 2^-21, and the accumulation
2^-24 of the sum of |r x| for every step of a row split: 3 per 8 rows (split) or
one per 2 rows (fp32 form).  Energies: 2^-20 of the sum of the rows' terms."""
import numpy as np
import pytest
import torch

from numpyro_amd import _lib

pytestmark = pytest.mark.gpu


def _data(N, D, C, seed, spread=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    X = torch.randn((N, D), generator=g, device="cuda")
    X[:, : D // 5] *= 10.0
    beta = 0.3 * torch.randn(D, generator=g, device="cuda") / D ** 0.5
    y = (torch.rand(N, generator=g, device="cuda") < torch.sigmoid(X @ beta)).float()
    z = beta + spread * 0.05 * torch.randn((C, D), generator=g, device="cuda")
    return X, y, z


def _stored(X, x_dtype):
    if x_dtype != "fp8":
        return X.double()
    m = X.abs().amax(0).double() / 448.0
    f, e = torch.frexp(m)
    s = torch.ldexp(torch.ones_like(m), torch.where(f == 0.5, e - 1, e))
    s = torch.where(m > 0, s, torch.ones_like(s))
    return (X / s.float()).to(torch.float8_e4m3fn).double() * s


def _eval(X, y, z, x_dtype, kernel):
    from numpyro_amd.infer.hmc import Engine
    from numpyro_amd.models import LogisticRegression
    C, D = z.shape
    eng = Engine(LogisticRegression(X, y, x_dtype=x_dtype, kernel=kernel), C, "NUTS", 0)
    pe = torch.full((C,), float("nan"), dtype=torch.float64, device="cuda")
    g = torch.full((C, D), float("nan"), device="cuda")
    torch.cuda.synchronize()
    _lib.check(_lib.load().nax_potential_grad(eng.h, _lib.ptr(z), D, C, _lib.ptr(pe),
                                              _lib.ptr(g)), "potential_grad")
    return pe, g.double()


def _check(X, y, z, x_dtype="fp32", kernel="mfma", chains=slice(None)):
    pe, g = _eval(X, y, z, x_dtype, kernel)
    pe, g, z64 = pe[chains], g[chains], z[chains].double()
    N, D = X.shape
    x = _stored(X, x_dtype)
    l = x @ z64.T
    r = torch.sigmoid(l) - y.double()[:, None]
    u = torch.nn.functional.softplus(l) - y.double()[:, None] * l
    want = r.T.contiguous() @ x + z64
    U = u.sum(0) + 0.5 * (z64 * z64).sum(1) + D * 0.5 * np.log(2 * np.pi)
    steps = N / 8  # rows of a split at least N / 256, 3 per 8 or 1 per 2 of them
    dr = 2.0 ** -21 + 0.25 * (D + 1) * 2.0 ** -24 * (x.abs() @ z64.abs().T)
    bound = dr.T.contiguous() @ x.abs() \
        + (2.0 ** -21 + steps * 2.0 ** -24) * (r.abs().T.contiguous() @ x.abs()) + 1e-6
    assert ((g - want).abs() <= bound).all()
    assert ((pe - U).abs() <= 2.0 ** -20 * u.abs().sum(0)).all()
    # and as a whole far inside it: rounding errors do not line up
    assert float((g - want).norm() / want.norm()) < 2e-5


@pytest.mark.parametrize("x_dtype, kernel", [("fp32", "mfma"), ("fp8", "auto")])
@pytest.mark.parametrize("D", [1, 7, 8, 31, 32, 33, 55, 64, 65, 96, 97, 128, 129, 161, 193, 225,
                               256])
def test_columns(D, x_dtype, kernel):
    _check(*_data(65536 + 31, D, 33, D), x_dtype=x_dtype, kernel=kernel)


@pytest.mark.parametrize("x_dtype, kernel", [("fp32", "mfma"), ("fp8", "auto")])
@pytest.mark.parametrize("N", [65535, 65536, 65537, 65568, 100003])
@pytest.mark.parametrize("C", [1, 32, 128, 129, 300])
def test_rows_and_chains(N, C, x_dtype, kernel):
    _check(*_data(N, 40, C, N + C), x_dtype=x_dtype, kernel=kernel)


@pytest.mark.parametrize("N, D, C", [(1, 3, 40), (31, 64, 5), (33, 200, 130), (5000, 90, 40)])
def test_few_rows_take_the_fp32_form(N, D, C):
    X, y, z = _data(N, D, C, N)
    _check(X, y, z)


def test_outlier_column_takes_the_fp32_form():
    X, y, z = _data(70000, 24, 40, 1, spread=0.1)
    X[17, 3] = 1e7  # far beyond 2^12 of the column's root mean square
    z[:, 3] = 1e-9
    _check(X, y, z)


@pytest.mark.parametrize("x_dtype, kernel", [("fp32", "mfma"), ("fp8", "auto")])
def test_non_finite_positions_stay_in_their_chain(x_dtype, kernel):
    X, y, z = _data(65600, 24, 40, 2)
    z[5, 2] = float("inf")
    z[6, 1] = float("nan")
    z[7, 0] = -3e38
    pe, _ = _eval(X, y, z, x_dtype, kernel)
    assert not torch.isfinite(pe[5:8]).any()
    keep = [c for c in range(40) if c not in (5, 6, 7)]
    _check(X, y, z, x_dtype=x_dtype, kernel=kernel, chains=keep)


@pytest.mark.parametrize("x_dtype", ["fp32", "fp8"])
def test_sampling_run_on_the_compacted_list(x_dtype):
    """Energies collected by a run (chains evaluated through the compacted
    list, in ever other groups) equal those of one evaluation of all chains
    at the same positions up to the order of the row splits (fp64 sums)."""
    from numpyro_amd import random as nrandom
    from numpyro_amd.infer import MCMC, NUTS
    from numpyro_amd.models import LogisticRegression
    X, y, z = _data(66000, 20, 150, 3, spread=0.1)
    model = LogisticRegression(X, y, x_dtype=x_dtype)
    mcmc = MCMC(NUTS(model, step_size=0.002), num_warmup=0, num_samples=4, num_chains=150)
    mcmc.run(nrandom.PRNGKey(4), init_params=z, extra_fields=("potential_energy", "num_steps"))
    draws = mcmc.get_samples(group_by_chain=True)["coefs"][:, -1].contiguous()
    pe, _ = _eval(X, y, draws, x_dtype, "auto")
    got = mcmc.get_extra_fields(group_by_chain=True)
    assert int(got["num_steps"].max()) > int(got["num_steps"].min())
    np.testing.assert_allclose(got["potential_energy"][:, -1].cpu().numpy(), pe.cpu().numpy(),
                               rtol=1e-12)
