"""Device memory that multishift solvers keep between solves: their work spinors,
given back when the solver is destroyed, when an allocation of the library would
fail without them, and at the end of a solve once all solvers together would keep
more than an eighth of the device's memory."""
import ctypes as C

import numpy as np
import pytest

import qphix_amd as q

pytestmark = pytest.mark.gpu

SHIFTS = [0.01 * 2 ** k for k in range(12)]


def memory():
    free, total = C.c_size_t(), C.c_size_t()
    h = C.CDLL("libamdhip64.so")
    assert h.hipDeviceSynchronize() == 0
    assert h.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value, total.value


def solve(s, g, b, x):
    try:
        s(x, b, SHIFTS[:len(x)], [1e-30] * len(x))
        raise AssertionError("converged")
    except q.QphixError as e:
        assert e.code == q.ENOCONV


def test_idle_solvers_give_their_work_spinors_back():
    g = q.Geometry([32, 32, 32, 32], q.F64, False)  # 101 MB a spinor
    M = q.Operator(g, q.OP_WILSON, q.gen_gauge(g, 8, 0.4), mass=0.3, t_boundary=-1.0)
    b = q.gen_spinor(g, 9, 1)
    x = [g.spinor() for _ in SHIFTS]
    solve(q.MInvCG(M, 3, 12), g, b, x)  # everything else is allocated and tuned
    want = [f.download(1) for f in x[:2]]
    before, total = memory()
    s = q.MInvCG(M, 3, 12)
    solve(s, g, b, x)
    kept = before - memory()[0]
    # 16 work spinors and the seven of a round of residuals
    assert kept <= 24 * g.bytes[0]
    # a request that no device can meet takes the idle solver's memory back
    # before it fails
    big = q.Geometry([128, 128, 128, 2046], q.F64, False)
    assert big.bytes[0] > total
    with pytest.raises(q.QphixError) as e:
        big.spinor()
    assert e.value.code == q.ENOMEM
    assert before - memory()[0] < 2 * g.bytes[0]
    # and it solves again
    solve(s, g, b, x)
    for f, w in zip(x, want):
        assert np.array_equal(f.download(1), w)
    del s
    assert before - memory()[0] < 2 * g.bytes[0]


def test_kept_work_spinors_are_bounded():
    g = q.Geometry([48, 48, 48, 64], q.F64, False)  # 680 MB a spinor, 16 GB a solver
    M = q.Operator(g, q.OP_WILSON, q.gen_gauge(g, 8, 0.4), mass=0.3, t_boundary=-1.0)
    b = q.gen_spinor(g, 9, 1)
    x = [g.spinor() for _ in SHIFTS]
    solvers = [q.MInvCG(M, 2, 12) for _ in range(4)]
    before, total = memory()
    for s in solvers:
        solve(s, g, b, x)
        assert before - memory()[0] <= total // 8
