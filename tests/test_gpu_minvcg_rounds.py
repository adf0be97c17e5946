"""Multishift CG applies the shifts' updates of eight iterations in one sweep
(FP64 and FP32): solves stopped after every number of iterations of a first,
second and third round, in device memory and replayed from graphs, against the
loop with host scalars, which updates them in each iteration: the same bits in
every solution. One solver object takes all solves, with more and fewer shifts in
turn (its work spinors change places), on parities that end inside a layout
block. Half storage keeps the sweep per iteration and is compared alike."""
import numpy as np
import pytest

import qphix_amd as q

pytestmark = pytest.mark.gpu

SHIFTS = [1e-3, 0.02, 0.5, 2.0]


def solve(s, g, b, n):
    xs = [g.spinor() for _ in range(n)]
    try:
        s(xs, b, SHIFTS[:n], [1e-30] * n)
        raise AssertionError("converged")
    except q.QphixError as e:
        assert e.code == q.ENOCONV
    return [x.download(1) for x in xs]


@pytest.mark.parametrize("latt", [[4, 4, 4, 4], [6, 4, 2, 10]])
@pytest.mark.parametrize("prec,c12", [(q.F64, False), (q.F32, True), (q.F16, True)])
def test_rounds_of_shift_updates(latt, prec, c12):
    g = q.Geometry(latt, prec, c12)
    M = q.Operator(g, q.OP_WILSON, q.gen_gauge(g, 8, 0.4), mass=0.3, t_boundary=-1.0)
    b = q.gen_spinor(g, 9, 1)
    for max_iters in list(range(2, 12)) + [16, 17, 18]:
        got = []
        for mode in (0, 1, 2):
            s = q.MInvCG(M, max_iters, len(SHIFTS), mode=mode)
            got.append([solve(s, g, b, n) for n in (2, 4, 3)])
        for other in got[1:]:
            for want, have in zip(got[0], other):
                for w, h in zip(want, have):
                    assert np.array_equal(w, h), max_iters
