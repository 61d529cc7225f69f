"""Device blocks kept for reuse behind nt_hip_alloc and nt_hip_free: blocks in use never overlap, at sizes
around every class edge; a block released and taken again carries the later work's data; a second free of
one block is an error of the next call; several threads may allocate and free."""
import ctypes as C
import threading

import numpy as np
import pytest

import noetic_ops as ops
import noetic_rl as nr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    nr.claim(0)
    yield


def alloc(n):
    p = C.c_void_p()
    assert nr.lib().nt_hip_alloc(n, C.byref(p)) == 0
    return p.value


def test_blocks_in_use_do_not_overlap():
    rng = np.random.default_rng(0)
    sizes = [1, 511, 512, 513, 576, 577] + [s + d for e in range(10, 22) for s in (1 << e, 9 << (e - 3), 15 << (e - 3))
                                            for d in (-1, 0, 1)]
    for _ in range(3):
        live = sorted((alloc(n), n) for n in rng.permutation(sizes))
        for (p, n), (q, _) in zip(live, live[1:]):
            assert p + n <= q
        for p, _ in live:
            nr.lib().nt_hip_free(p)
    big = alloc((128 << 20) + 1)  # past the largest kept block
    nr.lib().nt_hip_free(big)


def test_a_block_taken_again_holds_the_later_work():
    """Each round's tensors are released while the next round's are queued on the stream."""
    n = 300_000
    want, got = [], []
    for k in range(40):
        a = ops.fill((n,), float(k))
        b = ops.unary(ops.UnaryOp.ADD_SCALAR, a, ops.Layout([n]), 1.0)
        got.append(ops.reduce_all(ops.ReduceOp.MAX, b, n))
        want.append(k + 1.0)
        del a, b
    assert [float(g.to_numpy()[0]) for g in got] == want


def test_a_second_free_is_an_error():
    p = alloc(4096)
    nr.lib().nt_hip_free(p)
    nr.lib().nt_hip_free(p)
    assert nr.lib().nt_hip_sync() != 0
    assert nr.lib().nt_hip_sync() == 0
    a, b = alloc(4096), alloc(4096)
    assert a != b
    nr.lib().nt_hip_free(a)
    nr.lib().nt_hip_free(b)


def test_threads():
    bad = []

    def work(t):
        for i in range(60):
            n = 1000 + 37 * i + t
            x = ops.fill((n,), float(t * 1000 + i))
            if not (x.to_numpy() == t * 1000 + i).all():
                bad.append((t, i))

    ts = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
