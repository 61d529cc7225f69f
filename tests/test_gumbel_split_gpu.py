"""The Gumbel sampler's rows cut into several workgroups' segments, against Cpu(Reference)'s tokens for the
same stream: at the sizes where the number of segments changes, at every stream offset, with what decides
a row lying in one segment, and where segments' candidates tie or outnumber their slots."""
import numpy as np
import pytest

import noetic_rl as nr
from oracle import oracle as O

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module", autouse=True)
def device():
    nr.claim(0)
    yield


def both(x, tau, root, addmask=None, keep=None, pre_u32=0):
    m = nr.Tensor.from_numpy(addmask) if addmask is not None else None
    m = nr.Tensor.from_numpy(keep, "u8") if keep is not None else m
    rd, rc = nr.Rng(root, "split"), O.Rng(root, "split")
    for _ in range(pre_u32):
        rd.next_u32()
        rc.next_u32()
    dev = nr.sample_categorical(nr.Tensor.from_numpy(x), tau, m, rd).to_numpy().ravel().astype(np.int64)
    return dev, O.cpuref_sample_gumbel(x, tau, rc, addmask=addmask, keep=keep)


# one segment, two, several, 64 of them, a last one with a few blocks; rows that start inside a block
@pytest.mark.parametrize("rows,V", [(1, 1000), (1, 2040), (1, 2049), (1, 70000), (3, 5003), (16, 16391), (64, 4100),
                                    (128, 2055), (130, 2100)])
@pytest.mark.parametrize("tau,mask,pre", [(1.0, None, 0), (0.7, "u8", 1), (0.7, "f32", 6), (0.0, "u8", 0), (0.0, None, 3)])
def test_tokens_at_the_edges_of_segments(rows, V, tau, mask, pre):
    rng = np.random.default_rng(rows * V + pre)
    x = rng.normal(0, 2, (rows, V)).astype(F)
    keep = (rng.random((rows, V)) < 0.4).astype(np.uint8)
    keep[:, V // 2] = 1
    kw = {"keep": keep} if mask == "u8" else ({"addmask": np.where(keep, 0, -np.inf).astype(F)} if mask == "f32" else {})
    # (streams enough for some 60 rows; the two sides' f64 logarithms, rounded to f32, part once in 1e8 draws)
    for root in range(1 if tau == 0.0 else -(-60 // rows)):
        dev, cpu = both(x, tau, 7 + rows + 1000 * root, pre_u32=pre, **kw)
        np.testing.assert_array_equal(dev, cpu)


def test_what_decides_a_row_lies_in_one_segment():
    V = 20000
    x = np.random.default_rng(4).normal(0, 1, (6, V)).astype(F)
    keep = np.ones((6, V), np.uint8)
    keep[0] = 0
    keep[0, V - 1] = 1          # one token, in the last segment
    x[1, 3] = np.inf            # the row's maximum in the first
    x[2, :] = -np.inf
    x[2, 12345] = -3.0
    x[3, 5000:] = -np.inf       # segments with nothing allowed
    x[4, :V - 7] = -3e38        # a quotient by tau of -inf
    dev, cpu = both(x, 0.7, 3, keep=keep)
    np.testing.assert_array_equal(dev, cpu)
    assert dev[0] == V - 1 and dev[1] == 3 and dev[2] == 12345 and dev[4] >= V - 7
    for bad in (np.nan, "none"):
        y, k = x.copy(), keep.copy()
        if bad == "none":
            k[5] = 0
        else:
            y[5, 19000] = bad
        with pytest.raises(ValueError, match="position 5 has no allowed token"):
            both(y, 0.7, 3, keep=k)


@pytest.mark.parametrize("value,tau", [(1e7, 1.0), (-3e6, 0.7), (2e5, 1.0), (np.inf, 1.0)])
def test_ties_and_full_slots_over_segments(value, tau):
    """Logits so large that the sum's rounding makes ties across segments (the first wins), and more
    candidates within the margin than the slots hold (every element exactly)."""
    rng = np.random.default_rng(8)
    x = np.full((3, 9000), value, F)
    if np.isfinite(value):
        x[1] += rng.integers(0, 3, 9000).astype(F)
    dev, cpu = both(x, tau, 21)
    np.testing.assert_array_equal(dev, cpu)


@pytest.mark.parametrize("tau", [1e-45, 1e-40, 2.9e-39, 3e-39])
@pytest.mark.parametrize("rows,mask", [(260, None), (260, "u8"), (2, None)])
def test_temperatures_whose_reciprocal_overflows(tau, rows, mask):
    """Logits of the temperature's own size, several steps of each wave: their quotients are ordinary
    values although x (1 / tau) is infinite, and zeros' quotients are zeros."""
    V = 20000 if rows > 2 else 700_000
    rng = np.random.default_rng(rows)
    x = (rng.normal(-2, 2, (rows, V)) * tau).astype(F)
    x[1] = np.minimum(x[1], -F(1e-45))
    x[0, 5:] = 0.0
    if rows > 2:
        x[3] = -0.1  # quotients near -1e38 or -inf, and one row of them beside a zero in its last block
        x[3, V - 1] = 0.0
        x[4] = np.where(np.arange(V) % 7 == 0, F(0.25), x[4])  # overflows to +inf: the first of them
    keep = None
    if mask:
        keep = (rng.random((rows, V)) < 0.5).astype(np.uint8)
        keep[:, V - 1] = 1
    dev, cpu = both(x, tau, 17, keep=keep)
    np.testing.assert_array_equal(dev, cpu)


def test_a_temperature_that_is_zero_in_f32():
    """T = 1e-46 divides by an f32 zero: +inf for a positive logit, -inf for a negative one, a NaN (refused)
    for a zero."""
    x = np.full((3, 9000), -1.0, F)
    x[:, 8000] = x[:, 8500] = 2.0
    dev, cpu = both(x, 1e-46, 5)
    np.testing.assert_array_equal(dev, cpu)
    assert (dev == 8000).all()
    for value in (0.0, -2.0):  # row 1: 0 / 0, or nothing above -inf
        y = x.copy()
        y[1, 8000] = y[1, 8500] = value
        with pytest.raises(ValueError, match="position 1 has no allowed token"):
            both(y, 1e-46, 5)


def test_reruns_and_more_rows_agree():
    """A row's token does not depend on how the launch was cut: the first rows of a launch of 300 (one
    workgroup each) against the same rows alone."""
    x = np.random.default_rng(2).normal(0, 2, (300, 6000)).astype(F)
    many = nr.sample_categorical(nr.Tensor.from_numpy(x), 0.8, None, nr.Rng(9, "rows")).to_numpy()
    for n in (1, 4, 60, 200):
        few = nr.Tensor.from_numpy(np.ascontiguousarray(x[:n]))
        got = [nr.sample_categorical(few, 0.8, None, nr.Rng(9, "rows")).to_numpy() for _ in range(2)]
        np.testing.assert_array_equal(got[0], got[1])
        np.testing.assert_array_equal(got[0], many[:n])
