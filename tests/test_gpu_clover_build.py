"""The clover build kernel at the edges of its work-groups (64 sites): a
parity smaller than one, whole ones and a partial last one, in every output
kind and storage precision, against the oracle's blocks. Full complex blocks
are compared through their product with a Gaussian spinor. Tolerances are the
suite's: the relative rounding of the stored precision over a few roundings."""
import ctypes as C

import numpy as np
import pytest

import oracle
import qphix_amd as q

pytestmark = pytest.mark.gpu

MU, EPS, CSW, MASS = 0.013, 0.004, 1.0, 0.05
PRECS = [(q.F64, False, 1e-13), (q.F64, True, 1e-13), (q.F32, False, 2e-6), (q.F32, True, 2e-6),
         (q.F16, True, 5e-3), (q.BF16, True, 4e-2)]


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("latt", [[2, 2, 2, 2], [4, 4, 4, 4], [6, 4, 2, 10]])
@pytest.mark.parametrize("prec,c12,tol", PRECS)
def test_clover_build_matches_oracle(latt, prec, c12, tol):
    u = oracle.gen_gauge(latt, 31, 0.4)
    clov = oracle.clover_build(latt, u, CSW, MASS)
    g = q.Geometry(latt, prec, c12)
    ud = q.pack_gauge(g, u)
    for cb in (0, 1):
        half = clov[cb * g.vh * 72:(cb + 1) * g.vh * 72]
        up, dn, off = oracle.ndclover_inverse(half, MU, EPS)
        want = {q.CLOV_A: half, q.CLOV_AINV: oracle.clover_invert(half), q.CLOV_ND_OFF: off}
        for what, ref in want.items():
            got = q.clover_build(g, ud, CSW, MASS, cb, what, mu=MU, eps=EPS).download()
            assert rel(got, ref) < tol, (what, cb)
        psi = oracle.gen_spinor(latt, 7, cb)
        chi = g.spinor().upload(psi, cb)
        full = {q.CLOV_TMINV: oracle.full_clover_tm_inverse(half, MU), q.CLOV_ND_UP: up, q.CLOV_ND_DN: dn}
        for what, ref in full.items():
            f = q.clover_build(g, ud, CSW, MASS, cb, what, mu=MU, eps=EPS)
            res = g.spinor()
            q.call("qphix_clover_apply", g.h, res.p, chi.p, f.p, C.c_int(1))
            assert rel(res.download(cb), oracle.full_clover_apply(ref, psi)) < tol, (what, cb)
