"""Precision of the matrix-core kernel's forms (logit_split_kernel).

Small residuals in the matrix-core kernel's X^T R (logit_split_kernel): rare
events on one-hot and binary columns, where thousands of rows share one residual
far below 1 and an error of it has the same sign in all of them.

Reference: float64.  Bound of a gradient entry, relative to the sum of its |r x|: a
logit of K terms that are not zero carries K + 1 roundings, each at most 2^-24
of sum |x z| =: M; the exponential's argument a = |l| log2 e carries 1.5 roundings
2^-24 a, scaled by ln 2, and exp2, 1 + e, reciprocal and product together 6 of 2^-24;
the sums over a row split take 5 roundings per 32 rows (two products of R's grid
terms with each half tile, and the tile's fine terms), each at most 2^-24 of what
the split holds.  A split has at most 512 of the 131,072 rows.

Products in fp32: at z = 0 a residual is +-1/2, and a column with one number x that
is not zero has the gradient +-x/2 exactly; two fp16 terms of x miss its last bit
now and then."""
import math

import pytest
import torch

from numpyro_amd import _lib
from test_gpu_logistic_split import _check, _data, _stored

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


@pytest.mark.parametrize("x_dtype, C", [("fp32", 130), ("fp8", 33)])
@pytest.mark.parametrize("intercept", [-4.0, -7.0, -9.0])
def test_intercept_and_binary_columns(intercept, x_dtype, C):
    """Eight patterns of three binary columns beside an intercept; K = 4 terms of a
    logit are not zero."""
    g = torch.Generator(device="cuda").manual_seed(9)
    X = (torch.rand((N, 4), generator=g, device="cuda") < 0.3).float()
    X[:, 0] = 1.0
    beta = torch.tensor([intercept, 0.5, -0.7, 1.1], device="cuda")
    y = (torch.rand(N, generator=g, device="cuda") < torch.sigmoid(X @ beta)).float()
    z = beta + 0.1 * torch.randn((C, 4), generator=g, device="cuda")
    got = _grad(X, y, z, x_dtype, "auto")
    x, z64 = X.double(), z.double()
    l = x @ z64.T
    r = torch.sigmoid(l) - y.double()[:, None]
    want = r.T.contiguous() @ x + z64
    M = float((x @ z64.abs().T).max())
    eps = (5 * M + 1.5 * math.log(2) * 1.4427 * M + 6 + 5 * 512 / 32) * 2.0 ** -24
    bound = eps * (r.abs().T.contiguous() @ x) + 2.0 ** -23 * z64.abs() + 1e-9
    assert ((got - want).abs() <= bound).all(), float(((got - want).abs() / bound).max())


def _single_entries(C):
    """64 columns of one number each, 24 bits long, in rows of their own."""
    g = torch.Generator(device="cuda").manual_seed(5)
    X = torch.zeros((65536, 64), device="cuda")
    rows = torch.randperm(65536, generator=g, device="cuda")[:64]
    X[rows, torch.arange(64, device="cuda")] = 1 + torch.rand(64, generator=g, device="cuda")
    y = (torch.rand(65536, generator=g, device="cuda") < 0.5).float()
    want = (X[rows].amax(1) * (0.5 - y[rows])).double()
    return X, y, torch.zeros((C, 64), device="cuda"), want


def test_named_matrix_kernel_multiplies_in_fp32():
    X, y, z, want = _single_entries(40)
    assert torch.equal(_grad(X, y, z, "fp32", "mfma"), want.expand(40, 64))


@pytest.mark.parametrize("N, D, C", [(65536, 1, 129), (65537, 31, 130), (65567, 33, 130),
                                     (65568, 64, 300), (100003, 97, 129), (65537, 128, 130),
                                     (65537, 129, 130), (65537, 193, 129), (65569, 225, 130),
                                     (65537, 256, 300)])
def test_automatic_choice_at_the_edges_of_its_tiles(N, D, C):
    """Above 128 chains the automatic choice is the form in fp16 terms."""
    _check(*_data(N, D, C, N + D), kernel="auto")


@pytest.mark.filterwarnings("ignore:Out-of-support values")
@pytest.mark.parametrize("label", [4.5, -7.0, 1e6])
@pytest.mark.parametrize("x_dtype, C", [("fp32", 130), ("fp8", 33)])
def test_labels_outside_the_unit_interval(x_dtype, C, label):
    """A residual past fp16's range: the design takes the kernels in fp32.  Bound of
    a gradient entry: test_gpu_logistic_split's for a chain of fp32 multiply-adds."""
    X, y, z = _data(65600, 24, C, 6)
    y[1234] = label
    got = _grad(X, y, z, x_dtype, "auto")
    x, z64 = _stored(X, x_dtype), z.double()
    r = torch.sigmoid(x @ z64.T) - y.double()[:, None]
    want = r.T.contiguous() @ x + z64
    dr = 2.0 ** -21 + 0.25 * 25 * 2.0 ** -24 * (x.abs() @ z64.abs().T)
    bound = dr.T.contiguous() @ x.abs() \
        + (2.0 ** -21 + 65600 / 8 * 2.0 ** -24) * (r.abs().T.contiguous() @ x.abs()) + 1e-6
    assert ((got - want).abs() <= bound).all()


@pytest.mark.parametrize("label", [0.0, 1.0])
@pytest.mark.parametrize("lo, hi", [(-12.0, -6.0), (-6.0, -2.0), (-2.0, 0.0), (0.0, 2.0),
                                    (2.0, 6.0), (6.0, 12.0)])
def test_fp8_residuals_are_as_exact_as_the_tile_kernels(lo, hi, label):
    """Each of 64 columns has a 1 in one row, so that its gradient is that row's
    residual (the prior's part is 1e-12 of z).  250 x 64 residuals: their root mean
    square error from float64 varies by about 1 / sqrt(2 16000) = 0.6 % between samples
    of the same accuracy, hence 1.02."""
    from numpyro_amd.infer.hmc import Engine
    from numpyro_amd.models import LogisticRegression
    g = torch.Generator(device="cuda").manual_seed(8)
    X = torch.zeros((65536, 64), device="cuda")
    rows = torch.randperm(65536, generator=g, device="cuda")[:64]
    X[rows, torch.arange(64, device="cuda")] = 1.0
    y = torch.full((65536,), label, device="cuda")
    z = lo + (hi - lo) * torch.rand((250, 64), generator=g, device="cuda")
    want = torch.sigmoid(z.double()) if label == 0.0 else -torch.sigmoid(-z.double())
    err = {}
    for kernel in ("auto", "tile"):
        model = LogisticRegression(X, y, prior_scale=1e6, x_dtype="fp8", kernel=kernel)
        eng = Engine(model, 250, "NUTS", 0)
        pe = torch.empty(250, dtype=torch.float64, device="cuda")
        got = torch.empty((250, 64), device="cuda")
        torch.cuda.synchronize()
        _lib.check(_lib.load().nax_potential_grad(eng.h, _lib.ptr(z), 64, 250, _lib.ptr(pe),
                                                  _lib.ptr(got)), "potential_grad")
        err[kernel] = float((got.double() - 1e-12 * z.double() - want).square().mean().sqrt())
    assert err["auto"] <= 1.02 * err["tile"], err
