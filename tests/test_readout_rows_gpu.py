"""The readout fusion at the row counts where its first pass changes (32 and 64 rows) and at odd and short
k: the draws and their log-probabilities against the oracle on the logits, the logits against those of a
launch of 256 rows bit for bit, the recomputed block against the logits bit for bit."""
import numpy as np
import pytest

import noetic_rl as nr
from oracle import oracle as O

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module", autouse=True)
def device():
    nr.claim(0)
    prev = nr.set_matmul_precision(nr.MatmulPrecision.HALF)
    yield
    nr.set_matmul_precision(prev)


@pytest.mark.parametrize("d,V", [(16, 300), (128, 257), (144, 1000), (272, 2049)])
@pytest.mark.parametrize("masked", [False, True])
def test_rows_at_the_edges(d, V, masked):
    rng = np.random.default_rng(d + V)
    h = rng.normal(0, 1, (256, d)).astype(F)
    w = (rng.normal(0, 2, (d, V)) / np.sqrt(d)).astype(F)
    keep = (rng.random((256, V)) < 0.6).astype(np.uint8)
    keep[:, 0] = 1
    u = rng.random(256)
    W = nr.PackedReadout(nr.Tensor.from_numpy(w))

    def run(n, greedy=False):
        m = nr.Tensor.from_numpy(keep[:n], "u8") if masked else None
        t = nr.Tensor.from_numpy(h[:n])
        ut = nr.Tensor.from_numpy(u[:n], "f64")
        out = nr.readout_sample_logp(t, W, 0.0 if greedy else 0.7, m, None, uniforms=ut, debug=True)
        return [x.to_numpy() for x in out]

    full = run(256)
    for n in (1, 31, 32, 33, 64, 65):
        ids, lp, z, blk, at = run(n)
        np.testing.assert_array_equal(z.view(np.uint32), full[2][:n].view(np.uint32))
        t = O.tempered(z, 0.7, keep=keep[:n] if masked else None)
        want, edges = O.sample_invcdf(t, u[:n])
        assert not np.any((ids != want) & (edges >= 1e-6))
        np.testing.assert_allclose(lp, O.token_logp(t, ids), rtol=1e-5, atol=1e-6)
        for r in range(n):
            c = z[r, 32 * at[r]:32 * at[r] + 32]
            assert np.array_equal(blk[r, :c.size].view(np.uint32), c.view(np.uint32))
        g = run(n, greedy=True)[0]
        zz = np.where(keep[:n], z, -np.inf) if masked else z
        np.testing.assert_array_equal(g, zz.argmax(1))
