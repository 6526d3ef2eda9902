"""Operator application with a model's groups divided over several waves, at the
numbers of sources where the division changes (one wave task up to more than 2048)
and at term counts around the 64 terms and 64 groups a wave holds at a time.

The division changes neither the entries nor their order, so results of the same
sources in launches of different sizes are compared bit for bit; the oracle's sums
run in the same order (1e-12 for its own products).
"""

import numpy as np
import pytest

from oracle import applyop

pytestmark = pytest.mark.gpu


def _operator(n, n_terms, seed):
    """n_terms processes: number operators (one large group) and hoppings."""
    rng = np.random.default_rng(seed)
    op = {}
    kind = 0
    while len(op) < n_terms:
        i, j, k, l = (int(x) for x in rng.integers(n, size=4))
        proc = [((i, "c"), (i, "a")), ((i, "c"), (i, "a"), (j, "c"), (j, "a")), ((i, "c"), (j, "a")),
                ((i, "c"), (j, "c"), (k, "a"), (l, "a"))][kind % 4]
        kind += 1
        op.setdefault(proc, complex(rng.normal(), rng.normal()))
    return op


@pytest.mark.parametrize("n,n_terms", [(12, 1), (12, 63), (20, 64), (20, 65), (30, 400), (70, 129), (70, 400)])
def test_vector_apply_split(gpu, n, n_terms):
    from impuritymodel_amd.engine import Ops, vec_apply, vec_from_host
    from impuritymodel_amd.opcompile import n_words

    op = _operator(n, n_terms, 7 * n + n_terms)
    restr = {frozenset(range(0, n, 3)): (0, n // 4)}
    W = n_words(n)
    ops = Ops([op], [restr], n, W)
    rng = np.random.default_rng(n_terms)
    states = [int.from_bytes(rng.bytes(16), "big") >> (128 - n) for _ in range(2100)]

    def words(s):
        x = s << (64 * W - n)
        return [(x >> (64 * (W - 1 - w))) & (2**64 - 1) for w in range(W)]

    keys = [np.array([words(s)], np.uint64) for s in states]
    amp = [np.array([0.5 - 0.25j])] * len(states)

    def run(ids):
        v = vec_apply(ops, vec_from_host(W, [keys[i] for i in ids], [amp[i] for i in ids]),
                      np.arange(len(ids), dtype=np.int32), np.zeros(len(ids), np.int32), 1e-12)
        k, a, _ = v.get()
        k = np.asarray(k, np.uint64).reshape(-1, W)
        return [(k[v.offsets[i]:v.offsets[i + 1]], a[v.offsets[i]:v.offsets[i + 1]]) for i in range(len(ids))]

    full = run(range(2100))
    for i in (0, 5):
        ref = applyop.apply_op(n, op, {states[i]: 0.5 - 0.25j}, 1e-12, restr)
        assert [words(s) for s in ref] == full[i][0].tolist()
        np.testing.assert_allclose(full[i][1], list(ref.values()), rtol=0, atol=1e-12)
    for m in (1, 2, 63, 130, 1024, 2047, 2048):
        for i, (k, a) in enumerate(run(range(m))):
            assert np.array_equal(k, full[i][0]) and np.array_equal(a, full[i][1])


@pytest.mark.parametrize("fixed", [False, True])
@pytest.mark.parametrize("n_bath", [10, 50])
def test_build_split(gpu, n_bath, fixed):
    from impuritymodel_amd import finite
    from impuritymodel_amd.engine import Batch, Ops
    from impuritymodel_amd.models import make_model

    m = make_model(n_bath=n_bath, seed=3)
    n = m.n_spin_orbitals
    b = finite.get_basis(m.nBaths, m.nValBaths, m.dnValBaths, m.dnConBaths, m.dnTols, m.n0imps)
    seeds = finite._words(b[:130] if fixed else b[:3], n)
    ops = Ops([m.hOp], [m.restrictions], n)
    ref = None
    for copies in (1, 5, 33, 700):
        bt = Batch(ops, np.zeros(copies, np.int32))
        bt.set_seeds([seeds] * copies)
        bt.build(fixed_basis=fixed, weight_min=1e-12)
        rowptr, col, val = bt.csr()
        size = int(bt.chain_n[0])
        assert np.all(bt.chain_n == size)
        if ref is None:
            ref = rowptr, col, val, bt.basis_words()
        nnz = len(ref[1])
        assert np.array_equal(np.diff(rowptr).reshape(copies, size), np.tile(np.diff(ref[0]), (copies, 1)))
        assert np.array_equal(col.reshape(copies, nnz), np.tile(ref[1], (copies, 1)))
        assert np.array_equal(val.reshape(copies, nnz), np.tile(ref[2], (copies, 1)))
        assert np.array_equal(bt.basis_words(), np.tile(ref[3], (copies, 1)))


@pytest.mark.parametrize("vectors", [1, 100, 1 << 20])
@pytest.mark.parametrize("n_op,n_psi,size", [(1, 1, 1), (7, 3, 40), (3, 2, 0)])
def test_batched_memo_equals_one_by_one(gpu, monkeypatch, vectors, n_op, n_psi, size):
    """Transition states of all operators from one application against applyOp with a
    memo per operator, one state after the other: the same bits in the same order."""
    from impuritymodel_amd import finite, opcompile, spectra

    n = 20
    rng = np.random.default_rng(size)
    t_ops = [_operator(n, 5 + 3 * i, i) for i in range(n_op)]
    pool = [opcompile.words_to_bytes(np.array([[int(x) << (64 - n)]], np.uint64), n)[0]
            for x in rng.choice(1 << n, 60, replace=False)]
    psis = [{pool[i]: complex(*rng.normal(size=2)) for i in rng.permutation(60)[:size]} for _ in range(n_psi)]
    restr = {frozenset(range(8)): (1, 6)}
    ref = []
    for op in t_ops:
        memo = {}
        ref += [finite.applyOp(n, op, psi, 0.5, restr, memo) for psi in psis]
    monkeypatch.setattr(spectra, "_MEMO_VECTORS", vectors)
    keys, amps = spectra._transition_states_memo(n, t_ops, psis, 0.5, restr)
    assert len(keys) == len(amps) == len(ref)
    for k, a, r in zip(keys, amps, ref):
        assert opcompile.words_to_bytes(k, n) == list(r) and a.tolist() == list(r.values())
