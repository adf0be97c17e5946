"""Forced hop configurations hold on every lattice, the smallest included: the
work-group size of the launch itself, read from a captured graph's kernel node, is
the one asked for by qphix_tune_config(2, block, 0, 1) (natural site order) and by
qphix_set_hop_block without tuning, and the results are those of the default."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

import qphix_amd as q

pytestmark = pytest.mark.gpu

L = [4, 4, 4, 4]


class Dim3(C.Structure):
    _fields_ = [("x", C.c_uint), ("y", C.c_uint), ("z", C.c_uint)]


class KernelNodeParams(C.Structure):
    _fields_ = [("block", Dim3), ("extra", C.c_void_p), ("func", C.c_void_p), ("grid", Dim3), ("params", C.c_void_p),
                ("shared", C.c_uint)]


def blocks(work):
    """work-group sizes of the kernels that work() launches"""
    h = C.CDLL("libamdhip64.so")

    def ok(rc):
        assert rc == 0, rc

    stream, graph = C.c_void_p(), C.c_void_p()
    ok(h.hipStreamCreate(C.byref(stream)))
    try:
        q.set_stream(stream)
        ok(h.hipStreamBeginCapture(stream, 1))  # thread-local capture mode
        work()
        ok(h.hipStreamEndCapture(stream, C.byref(graph)))
        n = C.c_size_t(0)
        ok(h.hipGraphGetNodes(graph, None, C.byref(n)))
        nodes = (C.c_void_p * n.value)()
        ok(h.hipGraphGetNodes(graph, nodes, C.byref(n)))
        got = []
        for node in nodes:
            p = KernelNodeParams()
            ok(h.hipGraphKernelNodeGetParams(C.c_void_p(node), C.byref(p)))
            got.append(p.block.x)
        return got
    finally:
        q.set_stream(None)
        if graph.value:
            h.hipGraphDestroy(graph)
        h.hipStreamDestroy(stream)


def setup(prec, c12):
    g = q.Geometry(L, prec, c12)
    u = q.gen_gauge(g, 5, 0.4)
    return g, u[0], q.gen_spinor(g, 6, 1), q.gen_spinor(g, 7, 0), q.Dslash(g, t_boundary=-1.0)


@pytest.mark.parametrize("prec,c12", [(q.F64, False), (q.F32, True), (q.F16, True), (q.BF16, True)])
def test_forced_natural_order_holds_on_small_lattices(prec, c12):
    g, u, psi, chi, D = setup(prec, c12)
    outs = []
    try:
        for block in (None, 64, 128, 256):
            if block:
                q.call("qphix_tune_config", 2, block, 0, 1)
            a, b = g.spinor(), g.spinor()

            def work():
                D.dslash(a, psi, u, 1, 0)
                D.achimbdpsi(b, psi, chi, u, 4.1, 0.3, -1, 0)

            work()
            outs.append((a.download(0), b.download(0)))
            if block:
                assert blocks(work) == [block, block]
    finally:
        q.call("qphix_tune_config", 1, 256, 0, 1)
    for o in outs[1:]:
        assert np.array_equal(o[0], outs[0][0]) and np.array_equal(o[1], outs[0][1])


def set_block_child():
    g, u, psi, chi, D = setup(q.F32, True)
    a, b = g.spinor(), g.spinor()
    q.call("qphix_tune_config", 0, 256, 0, 1)
    D.dslash(a, psi, u, 1, 0)
    q.call("qphix_set_hop_block", 128)
    q.call("qphix_tune_config", 0, 256, 0, 1)
    assert blocks(lambda: D.dslash(b, psi, u, 1, 0)) == [128]
    D.dslash(b, psi, u, 1, 0)
    assert np.array_equal(a.download(0), b.download(0))


def test_work_group_size_holds_on_small_lattices():
    # in a process of its own: the size cannot be taken back
    subprocess.run([sys.executable, "-c", "from tests.test_gpu_tune_forced import set_block_child as c; c()"],
                   check=True, timeout=100,
                   cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
