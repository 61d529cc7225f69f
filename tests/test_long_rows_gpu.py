"""The general ops' paths for long rows, bit for bit: the last-axis sum in CpuRef's eight-partial order
with the row staged through LDS, the maximum with several loads in flight, and the binary ops over rows
against rows, a value per row or a scalar, aligned and not."""
import numpy as np
import pytest

import noetic_ops as ops
import noetic_rl as nr
from noetic_ops import BinaryOp, Layout, ReduceOp

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module", autouse=True)
def device():
    nr.claim(0)
    yield


def cpuref_sum(r):
    """kernels.rs:122-150: eight partials in order, folded pairwise, then the rest."""
    n8 = len(r) // 8 * 8
    p = np.zeros(8, F)
    for row in r[:n8].reshape(-1, 8):
        p = p + row
    acc = F(0)
    for k in range(4):
        acc = F(acc + F(p[k] + p[k + 4]))
    for v in r[n8:]:
        acc = F(acc + v)
    return acc


@pytest.mark.parametrize("n", [2047, 2048, 2049, 4095, 4096, 4103, 8192, 8200, 12287, 12288, 20488, 50304])
def test_sum_of_long_rows(n):
    rng = np.random.default_rng(n)
    x = (rng.standard_normal((5, n)) * np.exp(rng.standard_normal((5, n)) * 3)).astype(F)
    x[4, n // 2] = np.nan
    got = ops.reduce_dim(ReduceOp.SUM, nr.Tensor.from_numpy(x), (5, n), 1).to_numpy().ravel()
    want = np.array([cpuref_sum(r) for r in x], F)
    np.testing.assert_array_equal(got[:4].view(np.uint32), want[:4].view(np.uint32))
    assert np.isnan(got[4])
    assert ops.reduce_all(ReduceOp.SUM, nr.Tensor.from_numpy(x[0]), n).to_numpy()[0] == want[0]


@pytest.mark.parametrize("n", [1, 1024, 8191, 8192, 8193, 30001])
def test_first_maximum_of_long_rows(n):
    rng = np.random.default_rng(n)
    x = rng.integers(-50, 50, (6, n)).astype(F)  # ties
    x[1, n // 3] = np.nan
    x[2, n // 2:] = np.nan
    x[3] = -np.inf
    t = nr.Tensor.from_numpy(x)
    np.testing.assert_array_equal(ops.reduce_dim(ReduceOp.MAX, t, (6, n), 1).to_numpy().ravel(), x.max(1))
    np.testing.assert_array_equal(ops.reduce_dim(ReduceOp.ARGMAX, t, (6, n), 1).to_numpy().ravel(), x.argmax(1))


# a wave per row from 1024 rows of up to 4096, and from 4096 of up to 8192: both sides of each line, and
# rows shorter than a wave and than its eight loads
@pytest.mark.parametrize("rows,n", [(1024, 1), (1025, 63), (1027, 65), (1024, 511), (1023, 513), (1024, 4096), (1030, 4097),
                                    (4096, 8191), (4099, 8193), (70001, 9)])
def test_first_maximum_of_many_rows(rows, n):
    rng = np.random.default_rng(rows + n)
    x = rng.integers(-50, 50, (rows, n)).astype(F)  # ties
    x[1, n // 3] = np.nan
    x[2, n // 2:] = np.nan
    x[3] = -np.inf
    x[5, -1] = np.inf
    x[rows - 1, -1] = np.nan
    x[6], x[7] = 0.0, -0.0
    x[6, n // 2:] = -0.0  # equal zeros: the first one, sign and all
    t = nr.Tensor.from_numpy(x)
    at = x.argmax(1)
    np.testing.assert_array_equal(ops.reduce_dim(ReduceOp.ARGMAX, t, (rows, n), 1).to_numpy().ravel(), at)
    np.testing.assert_array_equal(ops.reduce_dim(ReduceOp.MAX, t, (rows, n), 1).to_numpy().ravel().view(np.uint32),
                                  x[np.arange(rows), at].view(np.uint32))


@pytest.mark.parametrize("op", list(BinaryOp))
@pytest.mark.parametrize("rows,cols,off", [(1, 1024, 0), (3, 1023, 0), (3, 1024, 0), (4, 4097, 0), (2, 5000, 1),
                                           (40000, 1028, 0)])
def test_binary_over_rows(op, rows, cols, off):
    rng = np.random.default_rng(cols + rows)
    f = {"ADD": np.add, "SUB": np.subtract, "MUL": np.multiply, "DIV": np.divide}[op.name]
    x = rng.standard_normal((rows, cols + off)).astype(F)
    y = rng.standard_normal((rows, cols + off)).astype(F)
    a, b = nr.Tensor.from_numpy(x), nr.Tensor.from_numpy(y)
    full = Layout([rows, cols], [cols + off, 1], off)
    col = Layout([rows, cols], [cols + off, 0], off)        # a value per row
    one = Layout([rows, cols], [0, 0], 0)                   # a scalar
    row = Layout([rows, cols], [0, 1], off)                 # one row against all
    X, Y = x[:, off:], y[:, off:]
    for al, bl, u, v in [(full, full, X, Y), (full, col, X, Y[:, :1]), (col, full, X[:, :1], Y),
                         (full, one, X, y[:1, :1]), (one, full, x[:1, :1], Y), (row, full, X[:1], Y), (col, row, X[:, :1], Y[:1])]:
        got = ops.binary(op, a, al, b, bl).to_numpy()
        np.testing.assert_array_equal(got.view(np.uint32), np.broadcast_to(f(u, v), X.shape).astype(F).view(np.uint32))


# both sides of each line between the two kernels, and last tiles that end at, before and past a group of 32
# values per chain
@pytest.mark.parametrize("rows,n", [(3, 4999), (3, 5000), (64, 4095), (64, 4096), (64, 4104), (64, 4344), (64, 4352), (64, 4361),
                                    (513, 8191), (520, 8200), (769, 16383), (1024, 16390), (1025, 16384)])
def test_sum_where_the_kernels_change(rows, n):
    rng = np.random.default_rng(rows + n)
    x = (rng.standard_normal((rows, n)) * np.exp(rng.standard_normal((rows, n)) * 3)).astype(F)
    x[0] = -0.0
    x[1, -1] = np.inf
    got = ops.reduce_dim(ReduceOp.SUM, nr.Tensor.from_numpy(x), (rows, n), 1).to_numpy().ravel()
    for r in [0, 1, 2, rows // 2, rows - 1]:
        assert got[r].view(np.uint32) == cpuref_sum(x[r]).view(np.uint32), r


@pytest.mark.parametrize("rows,cols", [(2048, 1030), (2049, 4100), (2047, 4100), (3, 4100), (2100, 1160)])
def test_one_row_against_many_of_little_over_a_workgroup(rows, cols):
    rng = np.random.default_rng(cols)
    x, y = rng.standard_normal((rows, cols)).astype(F), rng.standard_normal(cols).astype(F)
    a, b = nr.Tensor.from_numpy(x), nr.Tensor.from_numpy(y)
    full, row = Layout([rows, cols], [cols, 1], 0), Layout([rows, cols], [0, 1], 0)
    np.testing.assert_array_equal(ops.binary(BinaryOp.SUB, a, full, b, row).to_numpy(), x - y)
    np.testing.assert_array_equal(ops.binary(BinaryOp.SUB, b, row, a, full).to_numpy(), y - x)
