"""The half-precision product at the edges of its tiles, 64-k panels and routes: integer operands give the
exact product (every sum below 2^24 is an f32), in every orientation and at unaligned rows; the staged and
the packed path agree bit for bit on rounded operands; non-finite values stay in their rows and columns."""
import os

import numpy as np
import pytest

import noetic_rl as nr
from noetic_ops import DTensor, MatmulPrecision

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module", autouse=True)
def device():
    nr.claim(0)
    yield


def product(a, b, ta=False, tb=False, off=0):
    """a b from views: transposed storage, and rows that start `off` elements into a wider row."""
    def view(x, t):
        x = np.ascontiguousarray(x.T) if t else x
        wide = np.full((x.shape[0], x.shape[1] + off), 77.0, F)
        wide[:, off:] = x
        v = DTensor.from_numpy(wide).slice([range(0, x.shape[0]), range(off, x.shape[1] + off)])
        return v.swap_dims(0, 1) if t else v
    return view(a, ta).matmul_with(view(b, tb), MatmulPrecision.HALF).to_numpy()


@pytest.mark.parametrize("k", [1, 15, 63, 64, 65, 128, 191, 320])
@pytest.mark.parametrize("ta,tb,off", [(False, False, 0), (False, True, 1), (True, False, 3), (True, True, 0)])
def test_panels_and_tiles(k, ta, tb, off):
    rng = np.random.default_rng(k)
    for m, n in ((1, 1), (63, 65), (64, 64), (129, 31), (65, 200)):
        a, b = rng.integers(-16, 17, (m, k)).astype(F), rng.integers(-16, 17, (k, n)).astype(F)
        np.testing.assert_array_equal(product(a, b, ta, tb, off), a @ b)


@pytest.mark.parametrize("m,k,n", [(1537, 70, 1665), (2048, 130, 2048), (2500, 300, 2600)])
def test_large_tiles(m, k, n):
    rng = np.random.default_rng(m)
    a, b = rng.integers(-8, 9, (m, k)).astype(F), rng.integers(-8, 9, (k, n)).astype(F)
    np.testing.assert_array_equal(product(a, b), a @ b)


def test_staged_and_packed_agree():
    rng = np.random.default_rng(1)
    for m, k, n in ((300, 1000, 520), (1024, 333, 777)):
        a, b = rng.standard_normal((m, k)).astype(F), rng.standard_normal((k, n)).astype(F)
        got = []
        for path in ("staged", "packed"):
            os.environ["NOETIC_HIP_HALF_GEMM"] = path
            try:
                got.append(product(a, b))
            finally:
                del os.environ["NOETIC_HIP_HALF_GEMM"]
        np.testing.assert_array_equal(got[0].view(np.uint32), got[1].view(np.uint32))


def test_non_finite_values_stay_in_their_rows_and_columns():
    a, b = np.ones((70, 90), F), np.ones((90, 75), F)
    a[0, 5], a[69, 89], b[3, 0] = np.inf, np.nan, -np.inf
    got = product(a, b)
    assert (got[1:69, 1:] == 90).all()
    assert np.isnan(got[69]).all() and np.isnan(got[0, 0]) and (got[0, 1:] == np.inf).all()
    assert (got[1:69, 0] == -np.inf).all()
