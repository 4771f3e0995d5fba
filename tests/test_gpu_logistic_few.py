"""A few chains: the automatic choice at its edges.  Where the VALU tile kernel is the
faster one the results are its bits; on the other side of each edge the row tiles
are checked against float64 at theirs (32 rows, 64 columns, 4, 8 and 16 chains)."""
import pytest
import torch

from test_gpu_logistic_residuals import _grad
from test_gpu_logistic_rows import test_rows_against_float64 as check_rows
from test_gpu_logistic_split import _check, _data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x_dtype, N, D, C", [
    ("fp32", 1000, 256, 16), ("fp32", 3999, 65, 1), ("fp32", 500, 3, 31), ("fp32", 15999, 70, 9),
    ("fp32", 15999, 256, 31), ("fp32", 100001, 16, 17), ("fp8", 300001, 20, 1),
    ("fp8", 65536, 224, 8), ("fp8", 300001, 64, 16)])
def test_tile_kernel_where_it_is_faster(x_dtype, N, D, C):
    X, y, z = _data(N, D, C, N + D)
    assert torch.equal(_grad(X, y, z, x_dtype, "auto"), _grad(X, y, z, x_dtype, "tile"))


@pytest.mark.parametrize("x_dtype, N, D, C", [("fp32", 32001, 4, 17), ("fp32", 99999, 16, 31),
                                              ("fp8", 65536, 20, 1), ("fp8", 70001, 64, 16)])
def test_tile_kernel_at_half_the_row_splits(x_dtype, N, D, C):
    _check(*_data(N, D, C, N + D), x_dtype=x_dtype, kernel="auto")


@pytest.mark.parametrize("n, d, C", [(4000, 65, 1), (4033, 129, 8), (4127, 256, 5), (16000, 192, 9),
                                     (16001, 17, 31), (16031, 63, 20), (16385, 64, 17),
                                     (16000, 256, 31), (1048577, 1, 8)])
def test_row_tiles_from_the_edges_on(n, d, C):
    check_rows(n, d, C)


@pytest.mark.parametrize("N, D, C", [(65536, 225, 8), (65567, 225, 1), (65537, 65, 9),
                                     (70001, 33, 17)])
def test_fp8_matrix_cores_from_the_edges_on(N, D, C):
    X, y, z = _data(N, D, C, N + D)
    assert not torch.equal(_grad(X, y, z, "fp8", "auto"), _grad(X, y, z, "fp8", "tile"))
    _check(X, y, z, x_dtype="fp8", kernel="auto")
