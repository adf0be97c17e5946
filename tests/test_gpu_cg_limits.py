"""CG with iteration limits of 0, 1 and below 0 (which the host loop takes as no
iteration at all): statuses, counters, residuals and solutions of the device-scalar
modes equal those of the host-scalar mode, from a zero and a nonzero guess."""
import numpy as np
import pytest

import qphix_amd as q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["cg", "bicgstab"])
@pytest.mark.parametrize("max_iters", [-2, -1, 0, 1])
def test_iteration_limits_in_every_mode(kind, max_iters):
    g = q.Geometry([4, 4, 4, 4], q.F64, False)
    M = q.Operator(g, q.OP_WILSON, q.gen_gauge(g, 5, 0.4), mass=0.1, t_boundary=-1.0)
    b, x0 = q.gen_spinor(g, 6, 1), q.gen_spinor(g, 7, 1)
    for guess in (False, True):
        got = []
        for mode in (0, 1, 2):
            x = g.spinor()
            if guess:
                q.copy(g, x, x0)
            s = (q.InvCG if kind == "cg" else q.InvBiCGStab)(M, max_iters).set_mode(mode)
            st = s(x, b, 1e-12)
            got.append(((st.status, st.n_iters, st.rsd_sq_final, st.site_flops, st.mv_apps), x.download(1)))
        assert got[0][0][0] == q.ENOCONV
        for stats, x in got[1:]:
            assert stats == got[0][0]
            assert np.array_equal(x, got[0][1])
