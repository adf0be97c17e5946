"""Reductions of several streams in flight at once, and captured reductions
replayed beside eager ones: every stream and every capture counts and sums in
buffers of its own, so each result is the host form's (bit for bit), during the
overlap and after it. Also with more streams and captures than there are
buffers, one after the other."""
import ctypes as C

import numpy as np
import pytest

import qphix_amd as q

pytestmark = pytest.mark.gpu

# 1, 8, 135 and 2048 (the most) work-groups of a reduction
LATTICES = [[4, 4, 4, 4], [8, 8, 8, 8], [12, 12, 20, 24], [32, 32, 32, 32]]


class Hip:
    def __init__(self):
        h = C.CDLL("libamdhip64.so")
        vp, pp = C.c_void_p, C.POINTER(C.c_void_p)
        for name, args in {"hipMalloc": [pp, C.c_size_t], "hipFree": [vp], "hipMemcpy": [vp, vp, C.c_size_t, C.c_int],
                           "hipStreamCreateWithFlags": [pp, C.c_uint], "hipStreamDestroy": [vp],
                           "hipStreamSynchronize": [vp], "hipStreamBeginCapture": [vp, C.c_int],
                           "hipStreamEndCapture": [vp, pp], "hipDeviceSynchronize": [],
                           "hipGraphInstantiate": [pp, vp, vp, C.c_char_p, C.c_size_t], "hipGraphLaunch": [vp, vp],
                           "hipGraphExecDestroy": [vp], "hipGraphDestroy": [vp]}.items():
            fn = getattr(h, name)
            fn.argtypes = args
            setattr(self, name, self.checked(fn))
        self.streams, self.graphs, self.buffers = [], [], []

    @staticmethod
    def checked(fn):
        def run(*a):
            rc = fn(*a)
            assert rc == 0, (fn.__name__, rc)
        return run

    def stream(self):
        s = C.c_void_p()
        self.hipStreamCreateWithFlags(C.byref(s), 1)  # not ordered with the default stream
        self.streams.append(s)
        return s

    def doubles(self, n):
        p = C.c_void_p()
        self.hipMalloc(C.byref(p), 8 * n)
        self.buffers.append(p)
        return p.value

    def read(self, p, n):
        out = np.zeros(n)
        self.hipMemcpy(out.ctypes.data_as(C.c_void_p), C.c_void_p(p), 8 * n, 2)  # device to host
        return out

    def capture(self, stream, work):
        graph, exe = C.c_void_p(), C.c_void_p()
        q.set_stream(stream)
        self.hipStreamBeginCapture(stream, 1)  # thread-local capture mode
        work()
        self.hipStreamEndCapture(stream, C.byref(graph))
        self.hipGraphInstantiate(C.byref(exe), graph, None, None, 0)
        self.graphs.append((graph, exe))
        return exe

    def close(self):
        q.set_stream(None)
        self.hipDeviceSynchronize()
        for graph, exe in self.graphs:
            self.hipGraphExecDestroy(exe)
            self.hipGraphDestroy(graph)
        for s in self.streams:
            self.hipStreamDestroy(s)
        for p in self.buffers:
            self.hipFree(p)


@pytest.fixture
def hip():
    q.norm2(*field([4, 4, 4, 4], 1))  # the library is initialised
    h = Hip()
    yield h
    h.close()


def field(latt, seed):
    g = q.Geometry(latt, q.F64, False)
    return g, q.gen_spinor(g, seed, 1)


@pytest.fixture(scope="module")
def fields():
    out = []
    for k, latt in enumerate(LATTICES):
        g, x = field(latt, 3 + k)
        y = q.gen_spinor(g, 13 + k, 1)
        o = (C.c_double * 3)()
        q.call("qphix_inner_product_norm", g.h, x.p, y.p, o)
        out.append((g, x, y, q.norm2(g, x), list(o)))
    return out


def check_after(fields):
    q.set_stream(None)
    for g, x, y, n2, ip in fields:
        o = (C.c_double * 3)()
        q.call("qphix_inner_product_norm", g.h, x.p, y.p, o)
        assert q.norm2(g, x) == n2 and list(o) == ip


def test_streams_in_flight_at_once(hip, fields):
    rounds, n = 40, len(fields)
    streams = [hip.stream() for _ in range(n)]
    d = hip.doubles(4 * rounds * n)
    for r in range(rounds):
        for k in range(n):  # stream k takes the lattices in turn
            g, x, y, _, _ = fields[(k + r) % n]
            q.set_stream(streams[k])
            at = d + 32 * (r * n + k)
            q.reduce_dev("norm2_spinor", g, at, x)
            q.reduce_dev("inner_product_norm", g, at + 8, x, y)
    hip.hipDeviceSynchronize()
    got = hip.read(d, 4 * rounds * n).reshape(rounds, n, 4)
    for r in range(rounds):
        for k in range(n):
            _, _, _, n2, ip = fields[(k + r) % n]
            assert list(got[r, k]) == [n2] + ip, (r, k)
    check_after(fields)


def test_replays_beside_eager_reductions(hip, fields):
    a, b = hip.stream(), hip.stream()
    g, x, y, n2, ip = fields[3]
    d = hip.doubles(4)

    def work():
        q.reduce_dev("norm2_spinor", g, d, x)
        q.reduce_dev("inner_product_norm", g, d + 8, x, y)

    exe = hip.capture(a, work)
    for r in range(20):
        hip.hipGraphLaunch(exe, a)
        q.set_stream(b if r & 1 else a)
        for gs, xs, ys, ns, ips in fields:
            o = (C.c_double * 3)()
            q.call("qphix_inner_product_norm", gs.h, xs.p, ys.p, o)
            assert q.norm2(gs, xs) == ns and list(o) == ips, r
        hip.hipStreamSynchronize(a)
        assert list(hip.read(d, 4)) == [n2] + ip, r
    check_after(fields)


def test_more_streams_and_captures_than_buffers(hip, fields):
    n = 70
    d = hip.doubles(2 * n)
    graphs = []
    for k in range(n):
        g, x, _, _, _ = fields[k % 3]
        s = hip.stream()
        q.set_stream(s)
        q.reduce_dev("norm2_spinor", g, d + 8 * k, x)
        graphs.append((s, hip.capture(s, lambda: q.reduce_dev("norm2_spinor", g, d + 8 * (n + k), x))))
    for rep in range(3):
        for s, exe in graphs:
            hip.hipGraphLaunch(exe, s)
            hip.hipStreamSynchronize(s)
    hip.hipDeviceSynchronize()
    got = hip.read(d, 2 * n)
    want = [fields[k % 3][3] for k in range(n)]
    assert list(got[:n]) == want and list(got[n:]) == want
    check_after(fields)
