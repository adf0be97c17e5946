"""The hop form that splits the eight terms of a site over wavefronts, which
small lattices take, against the one that gives a work-item all of them (a
forced traversal selects it): the same bits for every kernel of the family,
storage precision and sign, with a twisted boundary and anisotropy, on parities
smaller than a work-group's 64 sites, of whole work-groups and with a partial
last one; and several sources in one launch against one at a time. (The split
form itself is compared with the oracle wherever the other tests use small
lattices.)"""
import numpy as np
import pytest

import qphix_amd as q

pytestmark = pytest.mark.gpu

PRECS = [(q.F64, False), (q.F64, True), (q.F32, False), (q.F32, True), (q.F16, True), (q.BF16, True)]


def family(D, o, p, chi, u, A, F, isign):
    D.dslash(o[0], p, u, isign, 0)
    D.achimbdpsi(o[1], p, chi, u, 4.1, 0.3, isign, 0)
    D.clov_dslash(o[2], p, u, A, isign, 0)
    D.clov_achimbdpsi(o[3], p, chi, u, A, 0.25, isign, 0)
    D.tm_dslash(o[4], p, u, isign, 0)
    D.tm_achimbdpsi(o[5], p, chi, u, 4.1, 0.25, isign, 0)
    D.tmclov_dslash(o[6], p, u, [F, F], isign, 0)
    return [f.download(0) for f in o]


@pytest.mark.parametrize("latt", [[2, 2, 2, 2], [4, 4, 4, 4], [6, 4, 2, 10]])
@pytest.mark.parametrize("prec,c12", PRECS)
def test_split_matches_one_work_item_per_site(latt, prec, c12):
    g64, g = q.Geometry(latt, q.F64, False), q.Geometry(latt, prec, c12)
    u64 = q.gen_gauge(g64, 21, 0.4)
    u = q.convert_gauge(g, g64, u64)[0]
    A = q.convert_clover(g, g64, q.clover_build(g64, u64, 1.0, 0.05, 0, q.CLOV_A))
    F = q.convert_clover(g, g64, q.clover_build(g64, u64, 1.0, 0.05, 0, q.CLOV_TMINV, mu=0.1), full=True)
    D = q.Dslash(g, t_boundary=-1.0, aniso_s=0.7, aniso_t=1.3, tbc=[None, complex(0.8, 0.6), None, None], mass=0.1,
                 twisted_mass=0.2, prec_mass_rho=0.05)
    p, chi = q.gen_spinor(g, 5, 1), q.gen_spinor(g, 6, 0)
    o = [g.spinor() for _ in range(7)]
    psis = [q.gen_spinor(g, 30 + r, 1) for r in range(3)]
    outs = [g.spinor() for _ in psis]
    try:
        for isign in (1, -1):
            q.call("qphix_tune_config", 1, 256, 0, 1)
            got = family(D, o, p, chi, u, A, F, isign)
            singles = []
            for x in psis:
                D.clov_dslash(o[0], x, u, A, isign, 0)
                singles.append(o[0].download(0))
            D.clov_dslash_multi(outs, psis, u, A, isign, 0)
            q.call("qphix_tune_config", 2, 256, 2, 1)  # tiles of two planes: one work-item per site
            want = family(D, o, p, chi, u, A, F, isign)
            for k, (a, b) in enumerate(zip(got, want)):
                assert np.array_equal(a, b), (isign, k)
            for a, b in zip(singles, outs):
                assert np.array_equal(a, b.download(0)), isign
    finally:
        q.call("qphix_tune_config", 1, 256, 0, 1)
