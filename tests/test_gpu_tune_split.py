"""The tuner keeps a site traversal for every hop kernel, also where the form with
the eight terms over wavefronts is the fastest for one source: launches that have no
such form (several sources, flavour doublets) use it."""
import re

import pytest

import qphix_amd as q

pytestmark = pytest.mark.gpu


def test_tuned_configurations_name_a_traversal():
    L = [16, 16, 32, 32]  # 131072 sites of a parity: tuned
    try:
        q.call("qphix_tune_config", 1, 256, 0, 1)
        for prec, c12 in ((q.F64, False), (q.F32, False), (q.F32, True), (q.F16, True)):
            g = q.Geometry(L, prec, c12)
            u = q.gen_gauge(g, 5, 0.4)
            D = q.Dslash(g, t_boundary=-1.0)
            psi, chi, o = q.gen_spinor(g, 6, 1), q.gen_spinor(g, 7, 0), g.spinor()
            for isign in (1, -1):
                D.dslash(o, psi, u[0], isign, 0)
                D.achimbdpsi(o, psi, chi, u[0], 4.1, 0.3, isign, 0)
                D.tm_dslash(o, psi, u[0], isign, 0)
        lines = [ln for ln in q.tune_summary().splitlines() if "16x16x32x32" in ln]
        assert len(lines) == 24
        for ln in lines:
            assert int(re.search(r" bz (-?\d+) ", ln).group(1)) >= 0, ln
    finally:
        q.call("qphix_tune_config", 1, 256, 0, 1)
