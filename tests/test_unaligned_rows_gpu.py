"""Rows of a length that is no multiple of eight, whose elements are loaded in vectors at their own
alignment and element by element only across the row's end: short rows, and rows one to eight elements
past a chunk, in every type and mask, against the oracle."""
import numpy as np
import pytest

import noetic_ops as ops
import noetic_rl as nr
from oracle import oracle as O

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module", autouse=True)
def device():
    nr.claim(0)
    yield


def on_device(x, dtype):
    t = nr.Tensor.from_numpy(x)
    t = t if dtype == "f32" else ops.cast(t, ops.Layout.contiguous(t.shape), dtype)
    return t, t.to_f64().astype(F)


@pytest.mark.parametrize("V", [1, 2, 7, 9, 15, 505, 511, 513, 518, 1031, 4097, 6151])
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("mask", [None, "u8", "f32"])
def test_sampler_scorer_and_backward(V, dtype, mask):
    rows, tau = 5, 0.7
    rng = np.random.default_rng(V)
    xt, x = on_device(rng.normal(0, 2, (rows, V)).astype(F), dtype)
    yt, y = on_device((x + rng.normal(0, 0.1, (rows, V))).astype(F), dtype)
    tok = rng.integers(0, V, rows).astype(np.int32)
    keep = (rng.random((rows, V)) < 0.7).astype(np.uint8)
    keep[np.arange(rows), tok] = 1
    add = np.where(keep, rng.normal(0, 0.2, (rows, V)), -np.inf).astype(F)
    kw = {None: {}, "u8": {"keep": keep}, "f32": {"addmask": add}}[mask]
    m = {None: None, "u8": nr.Tensor.from_numpy(keep, "u8"), "f32": nr.Tensor.from_numpy(add)}[mask]
    z, zr = O.tempered(x, tau, **kw), O.tempered(y, tau, **kw)
    u = rng.random(rows)
    ids, lp = nr.sample_logp(xt, tau, m, None, uniforms=nr.Tensor.from_numpy(u, "f64"))
    want, edges = O.sample_invcdf(z, u)
    assert not np.any((ids.to_numpy() != want) & (edges >= 1e-6))
    np.testing.assert_allclose(lp.to_numpy(), O.token_logp(z, ids.to_numpy()), rtol=1e-5, atol=1e-6)
    pol, ref, t = nr.Tempered(xt, tau, m), nr.Tempered(yt, tau, m), nr.Tensor.from_numpy(tok)
    logp, rlogp, kl, ent, stats = nr.score_with_stats(pol, ref, t)
    for got, w in ((logp, O.token_logp(z, tok)), (rlogp, O.token_logp(zr, tok)), (ent, O.entropy(z)), (kl, O.kl(z, zr))):
        np.testing.assert_allclose(got.to_numpy(), w, rtol=1e-5, atol=2e-6)
    g = [rng.normal(0, 1, rows).astype(F) for _ in range(3)]
    gt = [nr.Tensor.from_numpy(v) for v in g]
    grad = nr.score_grad(pol, ref, t, stats, kl=kl, entropy=ent, g_logp=gt[0], g_kl=gt[1], g_entropy=gt[2],
                         grad_dtype="f32")
    w = O.score_grad(z, tok, zr, *g) / F(tau)
    np.testing.assert_allclose(grad.to_numpy(), w, rtol=1e-4, atol=1e-6)
    half = nr.score_grad(pol, ref, t, stats, kl=kl, entropy=ent, g_logp=gt[0], g_kl=gt[1], g_entropy=gt[2],
                         grad_dtype="bf16")
    f = grad.to_numpy().view(np.uint32)
    np.testing.assert_array_equal(half.to_numpy(), ((f + 0x7FFF + ((f >> 16) & 1)) >> 16).astype(np.uint16))
