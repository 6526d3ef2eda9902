"""Grid-wide eigensolver with Gram-Schmidt passes only where the estimated
orthogonality needs them, against the same solver with two passes in every step
(eigen_dgks off) and against numpy.

Tolerances: eigenvalues carry eps |H| per step (2e-16 * 800 * a few hundred steps
< 1e-10); a converged pair's residual is at most tol max(1, |lambda|) = 1e-12 * 800
by the stopping rule plus that rounding, so 1e-9; vectors of separate eigenvalues
are orthogonal to residual over gap, 1e-9 / 1e-2.
"""

import numpy as np
import pytest
import scipy.sparse

pytestmark = pytest.mark.gpu


def _random_chain(n, complex_h, shift):
    rng = np.random.default_rng(n)
    d = min(1.0, 6.0 / n)

    def part():
        return scipy.sparse.random(n, n, density=d, random_state=rng, data_rvs=lambda k: rng.standard_normal(k)).toarray()

    a = part() + (1j * part() if complex_h else 0.0)
    return a + a.conj().T + np.diag(2.0 * rng.standard_normal(n) + shift)


@pytest.mark.parametrize("n,complex_h,shift", [(3, True, 0.0), (64, False, 0.0), (257, True, -700.0), (300, False, 5.0),
                                               (1200, False, -700.0), (1200, True, 0.0)])
def test_partial_reorthogonalization(gpu, n, complex_h, shift):
    from impuritymodel_amd import engine
    from impuritymodel_amd.engine import Batch, Ops

    h = _random_chain(n, complex_h, shift)
    hs = scipy.sparse.csr_matrix(h.astype(complex))
    b = Batch(Ops([{}], [None], 1), np.zeros(1, np.int32))
    b.set_csr([n], hs.indptr.astype(np.int64), hs.indices.astype(np.int32), hs.data)
    exact = np.linalg.eigvalsh(h)[:3]
    try:
        engine.set_tuning("flat_min_n", 0)
        ev, vecs, steps, ok = b.eigen(3, tol=1e-12)
        engine.set_tuning("eigen_dgks", 0)
        full_ev, _, full_steps, full_ok = b.eigen(3, tol=1e-12)
    finally:
        engine.set_tuning("flat_min_n", 32768)
        engine.set_tuning("eigen_dgks", 1)
    assert ok and full_ok and steps[0] == full_steps[0]
    assert np.abs(ev[0] - full_ev[0]).max() <= 1e-10
    assert np.abs(ev[0] - exact).max() <= 1e-10
    x = vecs.reshape(3, n)
    for k in range(3):
        assert np.linalg.norm(h @ x[k] - ev[0, k] * x[k]) <= 1e-9
    assert np.abs(x.conj() @ x.T - np.eye(3)).max() <= 1e-7


@pytest.mark.parametrize("n,complex_h,shift,width", [(1200, False, -700.0, 1.0), (900, True, -900.0, 1.0),
                                                     (1000, False, -900.0, 0.2), (700, True, 0.0, 1.0)])
@pytest.mark.parametrize("no_diagonal", [False, True])
def test_residuals_at_rounding(gpu, n, complex_h, shift, width, no_diagonal):
    """Steps past convergence, so that rounding alone is left of the residuals (products in extended
    precision): half an ulp of the energy on output and half of the diagonal on input, and 1e-13 for a
    spectrum of width 20 on a basis orthogonal to about 5e-15.  Rows without a diagonal entry make the
    width that of the energies: twice the residual with two passes in every step, and that ulp.  The
    vectors are orthogonal to rounding, 1e-14."""
    from impuritymodel_amd import engine
    from impuritymodel_amd.engine import Batch, Ops

    h = width * _random_chain(n, complex_h, shift / width)
    if no_diagonal:
        rows = np.arange(0, n, 3)  # rows without a stored diagonal entry
        h[rows, rows] = 0.0
    hs = scipy.sparse.csr_matrix(h.astype(complex))
    b = Batch(Ops([{}], [None], 1), np.zeros(1, np.int32))
    b.set_csr([n], hs.indptr.astype(np.int64), hs.indices.astype(np.int32), hs.data)
    exact = np.linalg.eigvalsh(h - shift * np.eye(n))[:3]
    coo = hs.tocoo()

    def solve():
        ev, vecs, _, _ = b.eigen(3, tol=0.0, max_steps=250, allow_noconv=True)
        x = vecs.reshape(3, n).astype(np.clongdouble)
        r = -ev[0][:, None].astype(np.longdouble) * x
        for k in range(3):
            np.add.at(r[k], coo.row, coo.data.astype(np.clongdouble) * x[k][coo.col])
        return ev[0], x.astype(complex), np.linalg.norm(r.astype(complex), axis=1)

    try:
        engine.set_tuning("flat_min_n", 0)
        ev, x, res = solve()
        engine.set_tuning("eigen_dgks", 0)
        _, _, full_res = solve()
    finally:
        engine.set_tuning("flat_min_n", 32768)
        engine.set_tuning("eigen_dgks", 1)
    ulp = np.spacing(np.abs(ev).max())
    print(n, complex_h, shift, width, no_diagonal, res, full_res, flush=True)
    assert res.max() <= 2 * full_res.max() + ulp
    if not no_diagonal:
        assert res.max() <= ulp + 1e-13
        assert np.abs((ev - shift) - exact).max() <= ulp + 1e-13
    assert np.abs(x.conj() @ x.T - np.eye(3)).max() <= 1e-14
