"""A solve that breaks down before its first iteration (a zero source) may be the
first user of a lattice's hop kernels: what the tuner then records are times of the
kernels at work, not of launches that skip themselves because the solve is over. The
links alone of 16x16x32x32 in FP64 (151 MB a launch) take 7 us at 20 TB/s, more than
anything beyond the caches' L2 delivers; a skipped launch takes less."""
import re

import pytest

import qphix_amd as q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [1, 2])
def test_zero_source_does_not_tune_on_skipped_launches(mode):
    L = [16, 16, 32, 32]  # 131072 sites of a parity: tuned
    g = q.Geometry(L, q.F64, False)
    M = q.Operator(g, q.OP_WILSON, q.gen_gauge(g, 5, 0.4), mass=0.1, t_boundary=-1.0)
    try:
        q.call("qphix_tune_config", 1, 256, 0, 1)
        st = q.InvBiCGStab(M, 100).set_mode(mode)(g.spinor(), g.spinor(), 1e-10)
        assert st.status == q.EBREAKDOWN
        M(g.spinor(), q.gen_spinor(g, 6, 1), 1, 1)  # tunes whatever the solve did not
        lines = [ln for ln in q.tune_summary().splitlines() if "16x16x32x32" in ln]
        assert len(lines) == 2
        bytes_moved = 144 * 8 * g.vh
        for ln in lines:
            assert float(re.search(r"([0-9.]+) ms$", ln).group(1)) * 1e-3 > bytes_moved / 20e12, ln
    finally:
        q.call("qphix_tune_config", 1, 256, 0, 1)
