"""Eigensolver on the register-resident basis (chains of up to 512 rows) and on
the basis in memory (larger chains), against numpy
at the edges of the launch classes, real and complex, alone and in batches that
change the number of waves per chain.

Tolerances: eigenvalues carry eps |H| per step (2e-16 * 800 * 600 steps = 1e-10 at
most, |H| < 800 here); a converged pair's residual is at most tol max(1, |lambda|)
= 1e-12 * 800 plus that rounding, so 1e-9.
"""

import numpy as np
import pytest
import scipy.sparse

pytestmark = pytest.mark.gpu


def _chain(n, complex_h, shift):
    rng = np.random.default_rng(100 + n)
    d = min(1.0, 6.0 / n)

    def part():
        return scipy.sparse.random(n, n, density=d, random_state=rng, data_rvs=lambda k: rng.standard_normal(k)).toarray()

    a = part() + (1j * part() if complex_h else 0.0)
    return a + a.conj().T + np.diag(2.0 * rng.standard_normal(n) + shift)


def _batch(hs):
    from impuritymodel_amd.engine import Batch, Ops

    ms = [scipy.sparse.csr_matrix(h.astype(complex)) for h in hs]
    rowptr = [0]
    for m in ms:
        rowptr.extend((m.indptr[1:] + rowptr[-1]).tolist())
    b = Batch(Ops([{}], [None], 1), np.zeros(len(ms), np.int32))
    return b.set_csr([m.shape[0] for m in ms], np.array(rowptr, np.int64),
                     np.concatenate([m.indices for m in ms]).astype(np.int32), np.concatenate([m.data for m in ms]))


@pytest.mark.parametrize("complex_h", [True, False])
@pytest.mark.parametrize("sizes,copies", [([1], 1), ([2, 3, 5, 17, 63, 64], 1), ([64, 40], 300), ([65, 100, 128], 1),
                                          ([90, 100], 260), ([129, 192], 1), ([193, 256], 1), ([257, 400], 1),
                                          ([512], 1), ([100, 513], 1), ([1100], 1), ([60, 2000], 150)])
def test_eigensolver_against_numpy(gpu, complex_h, sizes, copies):
    hs = [_chain(n, complex_h, -700.0 if n % 2 else 3.0) for n in sizes]
    b = _batch(hs * copies)
    ev, vecs, steps, ok = b.eigen(3, tol=1e-12)
    assert ok
    for i, h in enumerate(hs):
        n = len(h)
        exact = np.linalg.eigvalsh(h)[:3]
        k = len(exact)
        for c in {i, i + (copies - 1) * len(hs)}:
            assert 1 <= steps[c] <= n
            assert np.abs(ev[c, :k] - exact).max() <= 1e-10
            assert np.all(np.isnan(ev[c, k:]))
            base = int(b.row_base[c]) * 3
            x = vecs[base:base + 3 * n].reshape(3, n)
            assert not x[k:].any()
            for q in range(k):
                assert abs(np.linalg.norm(x[q]) - 1.0) <= 1e-12
                assert np.linalg.norm(h @ x[q] - ev[c, q] * x[q]) <= 1e-9


@pytest.mark.parametrize("n", [100, 700])
def test_eigensolver_reports_missed_tolerance(gpu, n):
    b = _batch([_chain(n, True, 0.0)])
    ev, _, steps, ok = b.eigen(3, tol=1e-12, max_steps=8, allow_noconv=True)
    assert not ok and steps[0] == 8
    assert np.all(np.isfinite(ev))


@pytest.mark.parametrize("complex_h", [True, False])
@pytest.mark.parametrize("n", [2, 40, 64, 100, 190, 256, 448])
def test_eigensolver_does_not_depend_on_the_batch(gpu, complex_h, n):
    """A chain on the register kernels has the same pairs, bit for bit, alone, among so many chains that
    the waves per chain change, beside chains whose launch it joins or that other kernels solve, and
    with the launch shapes of those kernels set by hand."""
    from impuritymodel_amd import engine

    h = _chain(n, complex_h, -700.0)
    small, empty = _chain(50, complex_h, 0.0), np.zeros((0, 0))
    batches = {"alone": [], "empty": [empty], "same": [_chain(n, complex_h, 3.0)], "joined": [_chain(500, complex_h, 0.0)],
               "memory": [_chain(600, complex_h, 0.0)], "wide": [_chain(1500, complex_h, 0.0), small],
               "many": [small] * 600, "most": [_chain(70, complex_h, 1.0)] * 2200}
    want = None

    def check(rest, name):
        nonlocal want
        b = _batch([h] + rest)
        ev, vecs, steps, ok = b.eigen(3, tol=1e-12)
        got = (ev[0], vecs[:3 * n], steps[0])
        want = want or got
        assert ok
        assert np.array_equal(got[0], want[0], equal_nan=True) and np.array_equal(got[1], want[1]), name
        assert got[2] == want[2], name

    for name, rest in batches.items():
        check(rest, name)
    try:
        for knob, value in (("eigen_bt", 256), ("eigen_bt", 512), ("eigen_bt", 1024), ("eigen_wave_max_n", 1024),
                            ("lanczos_lds_waves", 1), ("eigen_lds_vectors", 0)):
            engine.set_tuning(knob, value)
            check([], knob)
            check(batches["wide"], knob)
            engine.set_tuning(knob, {"eigen_bt": 0, "eigen_wave_max_n": 0, "lanczos_lds_waves": 4,
                                     "eigen_lds_vectors": -1}[knob])
    finally:
        for knob, value in (("eigen_bt", 0), ("eigen_wave_max_n", 0), ("lanczos_lds_waves", 4), ("eigen_lds_vectors", -1)):
            engine.set_tuning(knob, value)
