"""The doublet kernels that take both flavours in one launch, at the edges of
their work-groups (128 sites): parities smaller than one, whole ones and a
partial last one, against the single-flavour hops and passes they replace.
FP64 and FP32 results are the same bits (the same expressions, nothing rounded in
between); half storage skips the rounding of the hop results between the halves, so
it is held to the suite's tolerance of its precision."""
import ctypes as C

import numpy as np
import pytest

import qphix_amd as q

pytestmark = pytest.mark.gpu

MASS, MU, EPS = 0.1, 0.07, 0.03
PRECS = [(q.F64, False, 0.0), (q.F64, True, 0.0), (q.F32, False, 0.0), (q.F32, True, 0.0), (q.F16, True, 5e-3),
         (q.BF16, True, 4e-2)]


def same(got, want, tol):
    for a, b in zip(got, want):
        x, y = a.download(1), b.download(1)
        if tol == 0.0:
            assert np.array_equal(x, y)
        else:
            assert np.linalg.norm(x - y) < tol * np.linalg.norm(y)


@pytest.mark.parametrize("latt", [[2, 2, 2, 2], [4, 4, 4, 4], [6, 4, 2, 14]])
@pytest.mark.parametrize("prec,c12,tol", PRECS)
def test_doublet_operators_match_single_flavour_passes(latt, prec, c12, tol):
    g64, g = q.Geometry(latt, q.F64, False), q.Geometry(latt, prec, c12)
    u64 = q.gen_gauge(g64, 12, 0.4)
    u = q.convert_gauge(g, g64, u64)

    def term(cb, what, full=False, **kw):
        return q.convert_clover(g, g64, q.clover_build(g64, u64, 1.0, MASS, cb, what, **kw), full=full)

    A = term(1, q.CLOV_A)
    F = [term(0, w, True, mu=MU, eps=EPS) for w in (q.CLOV_ND_UP, q.CLOV_ND_DN)]
    off = term(0, q.CLOV_ND_OFF, mu=MU, eps=EPS)
    x = [q.gen_spinor(g, 3, 1), q.gen_spinor(g, 4, 1)]
    t, t2, y, z = ([g.spinor(), g.spinor()] for _ in range(4))
    al = 4.0 + MASS
    Mc = q.Operator(g, q.OP_NDTMCLOVER, u, clov=[None, A], fullclov=[F, None], clov_odiag=[off, None],
                    twisted_mass=MU, epsilon=EPS, t_boundary=-1.0)
    Mw = q.Operator(g, q.OP_NDTMWILSON, u, mass=MASS, twisted_mass=MU, epsilon=EPS, t_boundary=-1.0)
    D = q.Dslash(g, t_boundary=-1.0, mass=MASS, twisted_mass=MU, prec_mass_rho=MU)
    for isign in (1, -1):
        for f in range(2):
            D.dslash(t[f], x[f], u[0], isign, 0)
        D.two_flav_inverse_clover_term(t2, t, F, off, isign)
        for f in range(2):
            D.tmclov_achimbdpsi(z[f], t2[f], x[f], u[1], A, 0.25, isign, 1, f)
            q.call("qphix_axpy", g.h, C.c_double(-EPS), x[1 - f].p, z[f].p)
        Mc(y, x, isign, 1)
        same(y, z, tol)
        D.tmclov_two_flav_achimbdpsi(y, t2, x, u[1], A, 0.25, EPS, isign, 1)
        same(y, z, tol)
        mi = 1.0 / (al * al + MU * MU - EPS * EPS)
        q.call("qphix_two_flav_twisted_mass", g.h, (C.c_double * 2)(al * mi, -isign * MU * mi), C.c_double(EPS * mi),
               q._pa(t), q._pa(t2))
        for f in range(2):
            D.tm_achimbdpsi(z[f], t2[f], x[f], u[1], al, 0.25, isign, 1, 1.0 - 2.0 * f)
            q.call("qphix_axpy", g.h, C.c_double(-EPS), x[1 - f].p, z[f].p)
        Mw(y, x, isign, 1)
        same(y, z, tol)
        # a result in the place of an operand: the flavours one after the other
        for f in range(2):
            q.copy(g, y[f], x[f])
            q.copy(g, z[f], x[f])
        for f in range(2):
            D.tm_achimbdpsi(z[f], t2[f], z[f], u[1], al, 0.25, isign, 1, 1.0 - 2.0 * f)
            q.call("qphix_axpy", g.h, C.c_double(-EPS), z[1 - f].p, z[f].p)
        D.tm_two_flav_achimbdpsi(y, t2, y, u[1], al, 0.25, EPS, isign, 1)
        same(y, z, 0.0)
