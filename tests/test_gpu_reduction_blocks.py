"""Reductions end in the last work-group of their launch, which the groups of
64 work-groups count to: one work-group (no count), two, a whole group, one more
than a group, several groups and the largest launch of 2048. Every sum is taken
three times (the counters return to 0), by the host and the device form with
the same bits, against numpy. FP64 sums of at most 25 million positive terms,
at most 4096 of them one after the other, round by less than 1e-12 of their
value; the inner product is held to the same part of |l| |r|."""
import ctypes as C

import numpy as np
import pytest

import qphix_amd as q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("latt", [[4, 4, 4, 4], [8, 8, 8, 2], [8, 8, 8, 64], [10, 8, 8, 52], [16, 16, 16, 32],
                                  [32, 32, 32, 64]])
def test_reductions_over_any_number_of_work_groups(latt):
    g = q.Geometry(latt, q.F64, False)
    l, r = q.gen_spinor(g, 3, 1), q.gen_spinor(g, 4, 1)
    lh, rh = l.download(1), r.download(1)
    n2 = float(np.dot(lh, lh))
    dot = np.vdot(lh[0::2] + 1j * lh[1::2], rh[0::2] + 1j * rh[1::2])
    size = np.sqrt(n2 * float(np.dot(rh, rh)))
    dev = g.spinor()  # room for the device form's three results
    back = np.empty(3)
    first = None
    for _ in range(3):
        out = (C.c_double * 3)()
        q.call("qphix_inner_product_norm", g.h, l.p, r.p, out)
        assert abs(complex(out[0], out[1]) - dot) <= 1e-12 * size
        assert abs(out[2] - n2) <= 1e-12 * n2 and abs(q.norm2(g, l) - n2) <= 1e-12 * n2
        q.reduce_dev("inner_product_norm", g, dev.p, l, r)
        q.sync()
        assert C.CDLL("libamdhip64.so").hipMemcpy(back.ctypes.data_as(C.c_void_p), dev.p, C.c_size_t(24), 2) == 0
        assert list(back) == list(out)
        first = first or list(out)
        assert list(out) == first
