"""Device blocks kept for reuse behind nt_hip_alloc and nt_hip_free: blocks in use never overlap, at sizes
around every class edge; a block released and taken again carries the later work's data; a second free of
one block is an error of the next call; several threads may allocate and free; a block released while the
stream is captured is handed out to nobody, and no release becomes a node of the captured graph."""
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


class Capture:
    """What the library queues inside, as a graph."""

    def __init__(self):
        self.hip = C.CDLL("libamdhip64.so")
        self.stream, self.graph, self.exec = C.c_void_p(), C.c_void_p(), C.c_void_p()
        assert nr.lib().nt_hip_stream(C.byref(self.stream)) == 0

    def __enter__(self):
        assert self.hip.hipStreamBeginCapture(self.stream, 2) == 0  # (relaxed)
        return self

    def __exit__(self, *exc):
        rc = self.hip.hipStreamEndCapture(self.stream, C.byref(self.graph))
        assert exc[0] is not None or rc == 0

    def nodes(self):
        n = C.c_size_t()
        assert self.hip.hipGraphGetNodes(self.graph, None, C.byref(n)) == 0
        return n.value

    def replay(self):
        if not self.exec:
            assert self.hip.hipGraphInstantiate(C.byref(self.exec), self.graph, None, None, 0) == 0
        assert self.hip.hipGraphLaunch(self.exec, self.stream) == 0

    def close(self):
        if self.exec:
            self.hip.hipGraphExecDestroy(self.exec)
        self.hip.hipGraphDestroy(self.graph)


def test_a_block_released_during_a_capture_stays_the_graphs():
    n = 50_000
    x = nr.Tensor.from_numpy(np.arange(n, dtype=np.float32))
    held = alloc(4 * n)
    before = alloc(4 * n)
    lay = ops.Layout([n]).c()
    add = lambda src, dst: nr.lib().nt_hip_unary(int(ops.UnaryOp.ADD_SCALAR), 1.0, C.c_void_p(src),  # noqa: E731
                                                 C.byref(lay), C.c_void_p(dst))
    out, g = nr.Tensor((n,), "f32"), Capture()
    nr.sync()
    nr.lib().nt_hip_free(C.c_void_p(before))  # released before the capture, seen inside it
    with g:
        assert add(x.ptr, held) == 0 and add(held, out.ptr) == 0
        nr.lib().nt_hip_free(C.c_void_p(held))
        assert add(out.ptr, out.ptr) == 0  # (the next call takes the release in)
    assert g.nodes() == 3
    taken = [alloc(4 * n) for _ in range(8)]
    assert held not in taken and before in taken
    for _ in range(3):  # the program's own work on what it was given, between the replays
        for k, p in enumerate(taken):
            assert add(x.ptr, p) == 0
        g.replay()
        nr.sync()
        np.testing.assert_array_equal(out.to_numpy(), np.arange(n, dtype=np.float32) + 3)
        for p in taken:
            got = np.empty(n, np.float32)
            assert nr.lib().nt_hip_download(got.ctypes.data_as(C.c_void_p), C.c_void_p(p), 4 * n) == 0
            np.testing.assert_array_equal(got, np.arange(n, dtype=np.float32) + 1)
    assert nr.lib().nt_hip_free(C.c_void_p(held)) == 0  # a second release is still an error of the next call
    assert nr.lib().nt_hip_sync() != 0
    g.close()
    for p in taken:
        nr.lib().nt_hip_free(C.c_void_p(p))


def test_releases_past_the_limit_are_no_nodes_of_a_graph():
    """Six blocks of 128 MiB released before a capture and seen by the first call inside it: more than is
    kept. They go back to the device after it."""
    x, out, g = ops.fill((1000,), 1.0), nr.Tensor((1000,), "f32"), Capture()
    lay = ops.Layout([1000]).c()
    big = [alloc(128 << 20) for _ in range(6)]
    nr.sync()
    for p in big:
        nr.lib().nt_hip_free(C.c_void_p(p))
    with g:
        assert nr.lib().nt_hip_unary(int(ops.UnaryOp.ADD_SCALAR), 2.0, C.c_void_p(x.ptr), C.byref(lay),
                                     C.c_void_p(out.ptr)) == 0
    assert g.nodes() == 1
    for _ in range(3):
        g.replay()
        nr.sync()
        assert (out.to_numpy() == 3.0).all()
    g.close()
    again = [alloc(128 << 20) for _ in range(6)]
    for p in again:
        nr.lib().nt_hip_free(C.c_void_p(p))
    nr.sync()
