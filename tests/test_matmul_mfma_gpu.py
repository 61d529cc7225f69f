"""The f32 matmul's chains on the matrix cores: v_mfma_f32_32x32x2_f32 adds its two products in order,
each with one rounding, so every output has the bits of the oracle's fmaf chains
(oracle.c `or_matmul_f32`) on ordinary and on extreme operands, and at the edges of the tiles, of the
32-k panels and of the 256-k chains, in every orientation."""
import numpy as np
import pytest

import noetic_rl as nr
from noetic_ops import DTensor, MatmulPrecision
from oracle import oracle as O

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module", autouse=True)
def device():
    nr.claim(0)
    yield


def values(kind, shape, rng, is_a):
    x = rng.standard_normal(shape).astype(F)
    e = rng.integers(-20, 21, shape)
    if kind == "wide":
        return np.ldexp(x, e).astype(F)
    if kind == "subnormal products":
        return np.ldexp(x, (-70 if is_a else -66) + e // 4).astype(F)
    if kind == "subnormal operands":
        return rng.integers(0, 1 << 23, shape, dtype=np.uint32).view(F) * np.sign(x) if is_a else x
    if kind == "cancelling":
        return (np.ldexp(rng.integers(-1, 2, shape).astype(F), e) + np.ldexp(x, e - 22)).astype(F)
    if kind == "negative underflow":  # every product rounds a sum to -0
        return np.full(shape, -1e-30 if is_a else 1e-30, F)
    if kind == "specials":
        at = rng.integers(0, 300, shape)
        return np.select([at == 0, at == 1, at == 2, at == 3], [F(np.inf), F(-np.inf), F(0.0), F(-0.0)], x).astype(F)
    if kind == "overflow":
        return np.ldexp(x, 62 + e // 10).astype(F)
    return x


def same(got, want):
    """Bit for bit; a NaN for a NaN (their payloads are the instruction set's)."""
    n = np.isnan(want)
    return np.array_equal(n, np.isnan(got)) and np.array_equal(got.view(np.uint32)[~n], want.view(np.uint32)[~n])


def product(a, b, ta, tb):
    x = DTensor.from_numpy(np.ascontiguousarray(a.T) if ta else a)
    y = DTensor.from_numpy(np.ascontiguousarray(b.T) if tb else b)
    return (x.swap_dims(0, 1) if ta else x).matmul(y.swap_dims(0, 1) if tb else y).to_numpy()


@pytest.mark.parametrize("kind", ["normal", "wide", "subnormal products", "subnormal operands", "cancelling",
                                  "negative underflow", "specials", "overflow"])
def test_extreme_operands(kind):
    rng = np.random.default_rng(3)
    a, b = values(kind, (70, 301), rng, True), values(kind, (301, 90), rng, False)
    with np.errstate(all="ignore"):
        want = O.matmul(a, b)
    assert same(product(a, b, False, False), want), kind


@pytest.mark.parametrize("k", [1, 2, 31, 32, 33, 64, 255, 256, 257, 288, 513])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_panel_and_chain_edges(k, ta, tb):
    """64 tiles at one past, one short of and on their edge; the tail's padding keeps a -0."""
    rng = np.random.default_rng(k)
    for m, n in ((1, 1), (63, 65), (64, 64), (129, 31)):
        a, b = values("wide", (m, k), rng, True), values("wide", (k, n), rng, False)
        assert same(product(a, b, ta, tb), O.matmul(a, b)), (m, n)
    a, b = values("negative underflow", (3, k), rng, True), values("negative underflow", (k, 5), rng, False)
    got = product(a, b, ta, tb)
    assert same(got, O.matmul(a, b)) and np.signbit(got).all()


@pytest.mark.parametrize("m,k,n,ta,tb", [
    (1985, 40, 2049, False, False),   # 128 tiles, ragged on both sides
    (2048, 289, 2000, True, True),    # 128 tiles, two chains
    (65, 1100, 64, False, False),     # split k: five chains, the last one short
    (65, 1025, 64, True, True),       # split k, a last chain of one product
])
def test_tiles_and_splits(m, k, n, ta, tb):
    rng = np.random.default_rng(m + k)
    a, b = values("wide", (m, k), rng, True), values("wide", (k, n), rng, False)
    assert same(product(a, b, ta, tb), O.matmul(a, b))


@pytest.mark.parametrize("m,k,n", [(1, 300, 64), (64, 16, 1), (65, 40, 65), (128, 24, 64), (100, 32, 40), (3, 8, 5)])
@pytest.mark.parametrize("half", [False, True])
def test_many_small_batches(m, k, n, half):
    """Batches enough for 128 tiles, with sides that 64 tiles cover with less; a last panel of whole groups."""
    rng = np.random.default_rng(m + k)
    a, b = (rng.integers(-9, 10, (300,) + s).astype(F) for s in ((m, k), (k, n)))
    if not half:
        a *= F(1.1)
    got = DTensor.from_numpy(a).matmul_with(DTensor.from_numpy(b), MatmulPrecision.HALF if half else MatmulPrecision.F32)
    got = got.to_numpy()
    for z in (0, 1, 150, 299):
        assert same(got[z], a[z] @ b[z] if half else O.matmul(a[z], b[z])), z


@pytest.mark.parametrize("half", [False, True])
def test_more_batches_than_one_launch_holds(half):
    """17 million workgroups of 256 threads: over the 2^32 threads of a launch."""
    nb = 17_000_003
    a = DTensor.from_numpy((np.arange(nb) % 251).astype(F).reshape(nb, 1, 1))
    b = DTensor.from_numpy(np.full((1, 1, 1), 3, F))
    got = a.matmul_with(b, MatmulPrecision.HALF if half else MatmulPrecision.F32).to_numpy().ravel()
    np.testing.assert_array_equal(got, 3 * (np.arange(nb) % 251).astype(F))
