"""Gram matrices and combinations of sets of spinor fields at the edges of
their matrix-core tiles: set sizes around 4, 16 and the largest of 32, unequal
sets, one set against itself, parities smaller than a 64-site group and with
a partial last group, in FP64 and FP32, against numpy in FP64 on the stored
values. A sum of n products of unit-variance numbers rounds by less than
n eps / 2 in the storage precision (products and sums alike), the Gram sums of
FP32 by 256 eps over one word's sites before they go on in FP64."""
import numpy as np
import pytest

import oracle
import qphix_amd as q

pytestmark = pytest.mark.gpu

EPS = {q.F64: 2.0 ** -52, q.F32: 2.0 ** -23}


def fields(g, latt, n, seed):
    dev = [g.spinor().upload(oracle.gen_spinor(latt, seed + r, 1), 1) for r in range(n)]
    host = np.array([d.download(1) for d in dev])
    return dev, host[:, 0::2] + 1j * host[:, 1::2]


@pytest.mark.parametrize("latt", [[2, 2, 2, 2], [4, 4, 4, 8], [6, 4, 2, 10]])
@pytest.mark.parametrize("na,nb", [(1, 1), (3, 5), (4, 16), (16, 17), (17, 4), (31, 32), (32, 32)])
@pytest.mark.parametrize("prec", [q.F64, q.F32])
def test_gram_and_combine_sizes(prec, na, nb, latt):
    g = q.Geometry(latt, prec, False)
    a, ca = fields(g, latt, na, 500)
    b, cb = fields(g, latt, nb, 600)
    ref = ca.conj() @ cb.T
    scale = np.linalg.norm(ca, axis=1)[:, None] * np.linalg.norm(cb, axis=1)[None, :]
    assert np.abs(q.block_gram(g, a, b) - ref).max() <= (256 * EPS[prec] + 1e-13) * scale.max()
    same = q.block_gram(g, a, a)
    assert np.abs(same - ca.conj() @ ca.T).max() <= (256 * EPS[prec] + 1e-13) * scale.max()
    assert np.array_equal(same, same.conj().T)
    rng = np.random.default_rng(na * 100 + nb)
    m = rng.normal(size=(na, nb)) + 1j * rng.normal(size=(na, nb))
    y, cy = fields(g, latt, nb, 700)
    tol = 8 * (na + 1) * EPS[prec] * np.abs(m).max() * max(np.abs(ca).max(), np.abs(cy).max())
    out = [g.spinor() for _ in range(nb)]
    q.block_combine(g, a, m, None, out)  # no addend
    got = np.array([o.download(1) for o in out])
    assert np.abs(got[:, 0::2] + 1j * got[:, 1::2] - m.T @ ca).max() <= tol
    k = min(na, nb)
    q.block_combine(g, a, m, y, a[:k] + out[k:])  # outputs in the place of inputs
    got = np.array([o.download(1) for o in a[:k] + out[k:]])
    assert np.abs(got[:, 0::2] + 1j * got[:, 1::2] - (cy + m.T @ ca)).max() <= tol
