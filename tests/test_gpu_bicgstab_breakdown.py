"""BiCGStab breakdowns inside an iteration, in every control mode: <r0, M r0> = 0
(the zero operator) and |t|^2 = 0 (the identity: the first half step leaves no
residual, exactly). Statuses, counters and solutions equal those of the loop with
host scalars, and the solve ends there: with room for 20000 iterations it takes
less time than 400 iterations of a solve that does not break down."""
import time

import numpy as np
import pytest

import qphix_amd as q

pytestmark = pytest.mark.gpu

L = [4, 4, 4, 4]


def clover_op(g, u, diag):
    """res = diag * in: A = diag, A^-1 (of the other parity) = 0"""
    site = np.zeros((g.vh, 72))
    site[:, :12] = diag
    A = g.clover().upload(site.ravel())
    return q.Operator(g, q.OP_CLOVER, u, clov=[None, A], invclov=[g.clover(), None], t_boundary=-1.0)


def solve(M, g, b, mode, max_iters):
    best = 1e30
    for _ in range(3):
        x = g.spinor()
        s = q.InvBiCGStab(M, max_iters).set_mode(mode)
        q.sync()
        t = time.perf_counter()
        st = s(x, b, 1e-10)
        best = min(best, time.perf_counter() - t)
    return (st.status, st.n_iters, st.rsd_sq_final, st.site_flops, st.mv_apps), x.download(1), best


@pytest.mark.parametrize("prec,c12", [(q.F64, False), (q.F32, True), (q.F16, True), (q.BF16, True)])
def test_breakdown_inside_an_iteration_ends_the_solve(prec, c12):
    g = q.Geometry(L, prec, c12)
    u = q.gen_gauge(g, 5, 0.4)
    # real, equal entries: every product and sum of the identity's solve is exact
    ones = np.zeros((g.vh, 12, 2))
    ones[:, :, 0] = 1.0
    b = g.spinor().upload(ones.ravel(), 1)
    W = q.Operator(g, q.OP_WILSON, u, mass=0.1, t_boundary=-1.0)
    for diag in (0.0, 1.0):
        M = clover_op(g, u, diag)
        stats, x, _ = solve(M, g, b, 0, 20000)
        assert stats[0] == q.EBREAKDOWN and stats[1] == 1 and stats[4] == 2 + int(diag)
        for mode in (1, 2):
            got, xd, t = solve(M, g, b, mode, 20000)
            assert got == stats
            assert np.array_equal(xd, x)
            ref, _, t20 = solve(W, g, q.gen_spinor(g, 6, 1), mode, 20)
            assert t < 20 * t20, (diag, mode, t, t20)
