"""sort_desc around the sizes where its route changes (the run's threads and elements per thread, one
run or several, full and partial merge tiles), against the checker's stable order."""
import numpy as np
import pytest

import noetic_ops as ops
import noetic_rl as nr
from oracle import tensor_ops as T

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module", autouse=True)
def device():
    nr.claim(0)
    yield


def lanes(kind, shape, seed):
    rng = np.random.default_rng(seed)
    if kind == "normal":
        return rng.standard_normal(shape).astype(F)
    if kind == "ties":  # few values, both zeros, infinities
        return rng.choice(np.array([0.0, -0.0, 1.0, -1.0, np.inf, -np.inf, 1e-40], F), shape)
    if kind == "equal":
        return np.full(shape, -2.5, F)
    x = rng.integers(0, 1 << 32, shape, dtype=np.uint32).view(F)  # every bit pattern, NaNs of both signs among them
    return x


@pytest.mark.parametrize("n", [1, 2, 63, 65, 255, 256, 257, 1023, 1025, 4096, 4097, 8191, 8193, 16384, 16385, 18433,
                               32768, 32769, 49153])
@pytest.mark.parametrize("kind", ["normal", "ties", "equal", "bits"])
def test_values_and_positions(n, kind):
    outer, inner = (3, 1) if n > 300 else (5, 3)
    x = lanes(kind, (outer, n, inner), n)
    v, i = ops.sort_desc(nr.Tensor.from_numpy(x), (outer, n, inner))
    wv, wi = T.sort_desc(x, list(x.shape), 1)
    np.testing.assert_array_equal(i.to_numpy(), wi)
    np.testing.assert_array_equal(v.to_numpy().view(np.uint32), np.asarray(wv, F).view(np.uint32))


# the number of lanes also chooses the run's length (up to 64 long runs: a quarter) and the co-ranks'
# search (up to 512 merge tiles: a wave each): both sides of both, with partial last runs and tiles
@pytest.mark.parametrize("shape", [(32, 16385, 1), (33, 16385, 1), (1, 70001, 1), (64, 16389, 1), (8, 20480, 3),
                                   (29, 36865, 1)])
@pytest.mark.parametrize("kind", ["ties", "bits"])
def test_lane_counts(shape, kind):
    x = lanes(kind, shape, shape[1])
    v, i = ops.sort_desc(nr.Tensor.from_numpy(x), shape)
    wv, wi = T.sort_desc(x, list(shape), 1)
    np.testing.assert_array_equal(i.to_numpy(), wi)
    np.testing.assert_array_equal(v.to_numpy().view(np.uint32), np.asarray(wv, F).view(np.uint32))
