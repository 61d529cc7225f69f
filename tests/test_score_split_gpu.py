"""Rows scored by several workgroups (few rows of a large vocabulary), and the backward's steps spread
over several: against the oracle, bit for bit against the same rows in a launch of one workgroup per row, and
under capture, where the scorer keeps one workgroup per row."""
import ctypes as C

import numpy as np
import pytest

import noetic_rl as nr
from oracle import oracle as O

pytestmark = pytest.mark.gpu
F = np.float32
TOL = dict(rtol=1e-5, atol=1e-6)


@pytest.fixture(scope="module", autouse=True)
def device():
    nr.claim(0)
    yield


def rows_of(rows, V, seed, peak=False):
    rng = np.random.default_rng(seed)
    x = rng.normal(0, 1.5, (rows, V)).astype(F)
    if peak:
        x[:, V // 3] += 40.0
    y = (x + rng.normal(0, 0.1, (rows, V))).astype(F)
    keep = (rng.random((rows, V)) < 0.9).astype(np.uint8)
    tok = rng.integers(0, V, rows).astype(np.int32)
    keep[np.arange(rows), tok] = 1
    return x, y, keep, tok


# 1 to 64 segments per row; a last segment of one chunk; rows with nothing in some segments
@pytest.mark.parametrize("rows,V", [(1, 4096), (1, 4097), (1, 40001), (3, 16384), (16, 33000), (64, 8200), (65, 24600),
                                    (256, 13000)])
@pytest.mark.parametrize("masked,tau,peak", [(False, 1.0, False), (True, 0.7, False), (True, 1.0, True)])
def test_split_rows_against_the_oracle(rows, V, masked, tau, peak):
    x, y, keep, tok = rows_of(rows, V, rows + V, peak)
    mask = nr.Tensor.from_numpy(keep, "u8") if masked else None
    pol = nr.Tempered(nr.Tensor.from_numpy(x), tau, mask)
    ref = nr.Tempered(nr.Tensor.from_numpy(y), tau, mask)
    lp, rlp, kl, ent = nr.score(pol, ref, nr.Tensor.from_numpy(tok))
    zx, zy = (O.tempered(v, tau, keep=keep if masked else None) for v in (x, y))
    np.testing.assert_allclose(lp.to_numpy(), O.token_logp(zx, tok), **TOL)
    np.testing.assert_allclose(rlp.to_numpy(), O.token_logp(zy, tok), **TOL)
    np.testing.assert_allclose(ent.to_numpy(), O.entropy(zx), **TOL)
    np.testing.assert_allclose(kl.to_numpy(), O.kl(zx, zy), **TOL)


def scored(x, y, tok, tau, mask):
    """Every output and statistic of scoring rows x beside y, and logp and the entropy of x alone."""
    def put(v):
        return nr.Tensor.from_numpy(np.ascontiguousarray(v))
    m = None if mask is None else nr.Tensor.from_numpy(mask, "u8" if mask.dtype == np.uint8 else "f32")
    pol, ref, t = nr.Tempered(put(x), tau, m), nr.Tempered(put(y), tau, m), put(tok)
    lp, rlp, kl, ent, st = nr.score_with_stats(pol, ref, t)
    both = [lp, rlp, kl, ent, st.lse_base, st.lse_rest, st.ref_lse_base, st.ref_lse_rest]
    alone = nr.score(pol, None, t)
    return [v.to_numpy().ravel().view(np.uint32) for v in both], [alone[0].to_numpy().ravel().view(np.uint32),
                                                                  alone[3].to_numpy().ravel().view(np.uint32)]


# launches on both sides of 64 and 256 rows, rows of few chunks and of many, aligned and not; 270001 under an f32
# mask holds two batches per record
SHAPES = [(V, many, mask) for V, many in ((1000, 300), (8200, 300), (20001, 300), (50304, 600), (128256, 260))
          for mask in (None, "u8", "f32")] + [(270001, 258, "f32")]


@pytest.mark.parametrize("V,many,mask", SHAPES)
def test_a_rows_bits_do_not_depend_on_the_batch(V, many, mask):
    distinct = 24
    x, y, keep, tok = rows_of(distinct, V, V, peak=V % 2 == 0)
    if mask == "f32":  # one mask row shared by all; tokens that it keeps
        tok = np.flatnonzero(keep[0])[tok % int(keep[0].sum())].astype(np.int32)
    at = np.arange(many) % distinct

    def of(n):
        m = {"u8": keep[at[:n]], "f32": np.where(keep[:1], 0.0, -np.inf).astype(F), None: None}[mask]
        return scored(x[at[:n]], y[at[:n]], tok[at[:n]], 0.7 if mask else 1.0, m)

    want, alone = of(many)
    for a, w in zip(alone, (want[0], want[3])):
        np.testing.assert_array_equal(a, w)  # whether a reference is scored beside them or not
    for w in want:
        np.testing.assert_array_equal(w, w[:distinct][at])  # wherever the row stands
    for n in (1, 5, 64, 65, 130, 256):
        got, _ = of(n)
        for g, w in zip(got, want):
            np.testing.assert_array_equal(g, w[:n])


def test_masks_of_the_lowest_value():
    """An additive mask of the type's lowest finite value over whole batches of a row: weights of zero, and
    sums that stay finite."""
    V, rows = 40000, 6
    x, y, keep, tok = rows_of(rows, V, 12)
    keep[:, 9000:30000] = 0
    tok[:] = np.flatnonzero(keep[0])[:rows]
    add = np.where(keep[:1], 0.0, np.finfo(F).min).astype(F)
    mask = nr.Tensor.from_numpy(add)
    pol, ref = (nr.Tempered(nr.Tensor.from_numpy(v), 0.7, mask) for v in (x, y))
    lp, rlp, kl, ent = nr.score(pol, ref, nr.Tensor.from_numpy(tok))
    zx, zy = (O.tempered(v, 0.7, addmask=add) for v in (x, y))
    np.testing.assert_allclose(lp.to_numpy(), O.token_logp(zx, tok), **TOL)
    np.testing.assert_allclose(rlp.to_numpy(), O.token_logp(zy, tok), **TOL)
    np.testing.assert_allclose(ent.to_numpy(), O.entropy(zx), **TOL)
    np.testing.assert_allclose(kl.to_numpy(), O.kl(zx, zy), **TOL)


def test_refused_rows_and_infinities_in_some_segments():
    """A NaN in one segment refuses the row; a row allowed only in its last chunk is scored; one with
    nothing allowed is refused; +inf and -inf logits as in the unsplit kernel."""
    V, rows = 40960, 300
    x, _, _, tok = rows_of(rows, V, 9)
    keep = np.ones((rows, V), np.uint8)
    x[1, V - 5] = np.nan
    keep[2, : V - 3] = 0
    tok[2] = V - 1
    keep[3] = 0
    x[4, 100:30000] = -np.inf
    x[5, 7] = np.inf
    tok[6] = V
    for n in (8, 64):
        got = []
        for take in (n, rows):  # split, and one workgroup per row
            a = [nr.Tensor.from_numpy(np.ascontiguousarray(v[:take])) for v in (x, keep, tok)]
            out = [nr.Tensor((take,), "f32") for _ in range(4)] + [nr.Tensor((take,), "u8")]
            p = [t.ptr for t in out]
            args = nr.NtRlScoreArgs(a[0].ptr, None, nr.NT_F32, nr.NT_MASK_U8, take, V, V, a[1].ptr, V, 1.0, a[2].ptr, p[0],
                                    None, None, p[1], p[4], p[2], p[3], None, None, nr.NtMaskRows(0, 0, 0, 0))
            assert nr.lib().nt_hip_rl_score(C.byref(args)) == 0
            got.append([t.to_numpy()[:n] for t in out])
        np.testing.assert_array_equal(got[0][4], got[1][4])
        assert list(got[0][4][:8]) == [nr.NT_ROW_OK, nr.NT_ROW_NAN, nr.NT_ROW_OK, nr.NT_ROW_NO_TOKEN, nr.NT_ROW_OK,
                                       got[1][4][5], nr.NT_ROW_BAD_TOKEN, nr.NT_ROW_OK]
        for g, w in zip(got[0][:4], got[1][:4]):
            np.testing.assert_array_equal(g, w)


def test_capture_keeps_one_workgroup_per_row():
    """A captured call replays on another stream while the library's stream scores other rows, each
    replay with the eager call's bits."""
    hip = C.CDLL("libamdhip64.so")
    V, rows = 50000, 8
    x, _, _, tok = rows_of(rows, V, 5)
    z, _, _, tok2 = rows_of(rows, V, 6)

    def args(v, t):
        held = [nr.Tensor.from_numpy(v), nr.Tensor.from_numpy(t)] + [nr.Tensor((rows,), "f32") for _ in range(2)]
        return held, nr.NtRlScoreArgs(held[0].ptr, None, nr.NT_F32, nr.NT_MASK_NONE, rows, V, V, None, 0, 1.0,
                                      held[1].ptr, held[2].ptr, None, None, held[3].ptr, None, None, None, None, None,
                                      nr.NtMaskRows(0, 0, 0, 0))

    (ha, a), (hb, b) = args(x, tok), args(z, tok2)
    stream, other = C.c_void_p(), C.c_void_p()
    assert nr.lib().nt_hip_stream(C.byref(stream)) == 0  # (also frees what earlier tests released)
    assert hip.hipStreamCreateWithFlags(C.byref(other), 1) == 0
    graph, execu = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 2) == 0  # (relaxed)
    rc = nr.lib().nt_hip_rl_score(C.byref(a))
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0 and rc == 0
    assert hip.hipGraphInstantiate(C.byref(execu), graph, None, None, 0) == 0
    assert nr.lib().nt_hip_rl_score(C.byref(a)) == 0
    want = [t.to_numpy().tobytes() for t in ha[2:]]
    for _ in range(4):
        assert hip.hipGraphLaunch(execu, other) == 0
        assert nr.lib().nt_hip_rl_score(C.byref(b)) == 0
        assert hip.hipStreamSynchronize(other) == 0
        nr.sync()
        got = [t.to_numpy() for t in ha[2:]]
        np.testing.assert_allclose(got[0], O.token_logp(x, tok), **TOL)
        np.testing.assert_allclose(got[1], O.entropy(x), **TOL)
        np.testing.assert_allclose(hb[2].to_numpy(), O.token_logp(z, tok2), **TOL)
        assert want == [g.tobytes() for g in got]
    hip.hipGraphExecDestroy(execu)
    hip.hipGraphDestroy(graph)
    hip.hipStreamDestroy(other)


@pytest.mark.parametrize("rows,V", [(1, 4096), (1, 4104), (1, 12289), (7, 50000), (100, 20001)])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_backward_parts_cover_every_element_once(rows, V, dtype):
    """Each row's gradient equals the same row's in a launch of one workgroup per row, bit for bit."""
    x, y, _, tok = rows_of(rows, V, rows * 3 + V)
    many = -(-4097 // rows)  # copies of the rows until each takes one workgroup

    def grad(reps):
        def put(v):
            v = np.concatenate([v] * reps)
            t = nr.Tensor.from_numpy(v)
            if dtype == "f32" or v.ndim == 1:
                return t
            import noetic_ops as ops
            return ops.cast(t, ops.Layout.contiguous(t.shape), dtype)
        n = reps * rows
        pol, ref, tk = nr.Tempered(put(x), 1.0, None), nr.Tempered(put(y), 1.0, None), put(tok)
        st = nr.RowStats(*(nr.Tensor.from_numpy(np.tile(v, reps).astype(F)) for v in (lse, rest, rlse, rest)))
        g = [nr.Tensor.from_numpy(np.tile(np.linspace(-1, 1, rows).astype(F) + k, reps)) for k in range(4)]
        out = nr.score_grad(pol, ref, tk, st, kl=g[0], entropy=g[1], g_logp=g[2], g_kl=g[3], g_entropy=g[0])
        return out.to_numpy().reshape(n, V)[:rows]

    lse, rlse = O.token_logp(x, np.zeros(rows, np.int32)), O.token_logp(y, np.zeros(rows, np.int32))
    lse, rlse, rest = x[:, 0] - lse, y[:, 0] - rlse, np.zeros(rows)
    if rows * V * many > 60_000_000:
        many = 60_000_000 // (rows * V)
        assert 4096 // (rows * many) < 4096 // rows
    np.testing.assert_array_equal(grad(1), grad(many))
