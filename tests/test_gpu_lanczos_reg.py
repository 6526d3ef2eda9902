"""Register-resident Lanczos (reorth = 1, chains of up to 1024 rows) against a
numpy recurrence with two Gram-Schmidt passes per step, at the edges of its
launch classes (64-row steps, one to four rows per thread), with bases that fit
the registers, that reach into LDS and that reach into memory, for complex,
real and imaginary start vectors and with enough chains to change the number of
waves per chain.

Tolerance: the two recurrences differ by rounding only; full
reorthogonalization keeps the amplification of a step's rounding (about
eps |H| sqrt(n) = 1e-13 here) at the level of the step count, so 1e-10 of |H|
leaves more than a factor of four at 200 steps.
"""

import numpy as np
import pytest
import scipy.sparse

pytestmark = pytest.mark.gpu


def _lanczos(h, v, K):
    V, alpha, beta = [v], [], []
    w = h @ v
    for j in range(min(K, len(v))):
        alpha.append(np.vdot(w, V[-1]).real)
        if j + 1 == min(K, len(v)):
            break
        w = w - alpha[-1] * V[-1] - (beta[-1] * V[-2] if j else 0.0)
        for _ in range(2):
            m = np.array(V)
            w = w - m.T @ (m.conj() @ w)
        beta.append(np.linalg.norm(w))
        V.append(w / beta[-1])
        w = h @ V[-1]
    return np.array(alpha), np.array(beta)


def _chain(rng, n, complex_h, start):
    def part():
        return scipy.sparse.random(n, n, density=min(1.0, 5.0 / n), random_state=rng,
                                   data_rvs=lambda k: rng.standard_normal(k)).toarray()

    a = part() + (1j * part() if complex_h else 0.0)
    h = a + a.conj().T + np.diag(3.0 * rng.standard_normal(n))
    v = rng.standard_normal(n) + (1j * rng.standard_normal(n) if start == "complex" else 0.0)
    v = 1j * v if start == "imaginary" else v
    return scipy.sparse.csr_matrix(h.astype(complex)), v / np.linalg.norm(v)


def _built(chains):
    from impuritymodel_amd.engine import Batch, Ops

    b = Batch(Ops([{}], [None], 1), np.zeros(len(chains), np.int32))
    rowptr = [0]
    for h, _ in chains:
        rowptr.extend((h.indptr[1:] + rowptr[-1]).tolist())
    b.set_csr([h.shape[0] for h, _ in chains], np.array(rowptr, np.int64),
              np.concatenate([h.indices for h, _ in chains]).astype(np.int32),
              np.concatenate([h.data for h, _ in chains]))
    return b


def _run(chains, K):
    return _built(chains).lanczos(K, reorth=1, v0=np.concatenate([v for _, v in chains]))


@pytest.mark.parametrize("complex_h,start", [(True, "complex"), (False, "complex"), (False, "real"),
                                             (False, "imaginary")])
@pytest.mark.parametrize("sizes,K,copies", [
    ([1, 2, 3, 36, 37, 63, 64], 64, 1),     # one wave of rows, many waves per chain
    ([60, 64], 64, 600),                    # one wave per chain, basis in registers and LDS
    ([65, 128], 128, 1),
    ([97, 128], 128, 150),
    ([129, 192], 192, 1),
    ([193, 256], 150, 2),
    ([257, 512], 90, 1),                    # two rows per thread, basis into memory
    ([513, 768], 60, 1),
    ([769, 1024], 50, 1),
    ([1024], 200, 1),
])
def test_register_lanczos_matches_numpy(gpu, complex_h, start, sizes, K, copies):
    rng = np.random.default_rng(5)
    chains = [_chain(rng, n, complex_h, start) for n in sizes]
    alpha, beta, kout, status = _run(chains * copies, K)
    for i, (h, v) in enumerate(chains):
        a, b = _lanczos(h, v, K)
        scale = max(1.0, abs(h).sum(axis=1).max())
        for c in range(i, len(chains) * copies, len(chains)):
            assert (kout[c], status[c]) == (min(K, len(v)), 0)
            assert np.abs(alpha[c, : len(a)] - a).max() <= 1e-10 * scale
            assert np.abs(beta[c, : len(b)] - b).max(initial=0.0) <= 1e-10 * scale


def test_register_lanczos_breakdown_and_empty_chain(gpu):
    # an eigenvector of a diagonal H as start vector: beta_0 is exactly zero
    from impuritymodel_amd._lib import IMPED_ERR_BREAKDOWN

    h = scipy.sparse.diags(np.arange(1.0, 6.0)).tocsr().astype(complex)
    e = np.zeros(5, complex)
    e[2] = 1.0
    rng = np.random.default_rng(6)
    other = _chain(rng, 70, True, "complex")
    alpha, _, kout, status = _run([(h, e), other, (scipy.sparse.csr_matrix((0, 0), dtype=complex), e[:0])], 10)
    assert (kout[0], status[0], alpha[0, 0]) == (1, IMPED_ERR_BREAKDOWN, 3.0)
    assert (kout[1], status[1]) == (10, 0)
    assert (kout[2], status[2]) == (0, 0)


@pytest.mark.parametrize("complex_h", [True, False])
@pytest.mark.parametrize("n_empty,others", [(1, 0), (3, 0), (1, 300), (2, 300)])
def test_register_lanczos_launch_of_empty_chains_only(gpu, complex_h, n_empty, others):
    # no state in any chain of a launch: alone, and beside more chains of 70 rows
    # than the chip has CUs (the classes then launch separately)
    empty = (scipy.sparse.csr_matrix((0, 0), dtype=complex), np.zeros(0, complex))
    chain = _chain(np.random.default_rng(7), 70, complex_h, "complex" if complex_h else "real")
    alpha, _, kout, status = _run([empty] * n_empty + [chain] * others, 12)
    assert not kout[:n_empty].any() and not status[:n_empty].any()
    if others:
        a, _ = _lanczos(*chain, 12)
        assert (kout[n_empty:] == 12).all() and not status[n_empty:].any()
        scale = max(1.0, abs(chain[0]).sum(axis=1).max())
        assert np.abs(alpha[n_empty:] - a).max() <= 1e-10 * scale


@pytest.mark.parametrize("complex_h,start", [(True, "complex"), (False, "complex"), (False, "real"),
                                             (False, "imaginary")])
@pytest.mark.parametrize("n,K", [(40, 40), (64, 64), (100, 100), (150, 80), (225, 150), (300, 90), (600, 60), (900, 40)])
def test_register_lanczos_does_not_depend_on_the_batch(gpu, complex_h, start, n, K):
    """The same bits alone, among so many chains that the waves per chain change, beside a chain
    whose launch it joins, with fewer waves by hand, and, for a real H, in the complex arithmetic
    that a complex chain in the batch brings."""
    from impuritymodel_amd import engine

    rng = np.random.default_rng(n)
    chain = _chain(rng, n, complex_h, start)
    wide = _chain(rng, n, complex_h, start)  # rows longer than the entries kept in registers
    dense = scipy.sparse.random(n, n, density=0.3, random_state=rng).tocsr()
    wide = ((wide[0] + (dense + dense.T)).tocsr(), wide[1])
    others = {"alone": [], "pair": [_chain(rng, n, complex_h, start)], "larger": [_chain(rng, 1000, complex_h, "real")],
              "middle": [_chain(rng, 260, complex_h, "complex")], "complex": [_chain(rng, 30, True, "complex")],
              "many": [_chain(rng, 33, complex_h, start)] * 600, "most": [_chain(rng, 65, complex_h, start)] * 2200}
    for c in (chain, wide):
        want = None
        for name, rest in others.items():
            alpha, beta, kout, status = _run([c] + rest, K)
            got = (alpha[0, :kout[0]], beta[0, :kout[0] - 1])
            assert (kout[0], status[0]) == (min(K, n), 0), name
            want = want or got
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), name
        try:
            for waves in (1, 2):
                engine.set_tuning("lanczos_lds_waves", waves)
                alpha, beta, kout, _ = _run([c], K)
                assert np.array_equal(alpha[0, :kout[0]], want[0]) and np.array_equal(beta[0, :kout[0] - 1], want[1])
        finally:
            engine.set_tuning("lanczos_lds_waves", 4)
