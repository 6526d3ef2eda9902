"""Continued fractions with a spectrum's chains side by side, at the edges of the
64-energy workgroups and of the numbers of chains per wave, against the kernel that
sums them one after the other (the same launch padded with empty spectra until it
fills the chip): the same bits, since the sum runs in the same order.

Against numpy: each level adds a few roundings of relative size 2e-16 and |g| stays
below 1 / delta = 10, so 100 levels stay within 1e-12 of the chain's own scale;
1e-10 of the largest value leaves room for cancellation in the sums.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chains", [1, 2, 3, 9, 16, 17, 40])
@pytest.mark.parametrize("n,n_w", [(1, 1), (6, 63), (90, 64), (90, 65), (30, 401)])
def test_split_equals_unsplit(gpu, chains, n, n_w):
    from impuritymodel_amd.engine import Batch, Ops

    rng = np.random.default_rng(1000 * chains + n)
    rowptr, col, val = [0], [], []
    for c in range(chains):
        for i in range(n):
            for j in (i - 1, i, i + 1):
                if 0 <= j < n:
                    col.append(j)
                    val.append(1.0 + min(i, j) % 3 if i != j else rng.normal())
            rowptr.append(len(col))
    b = Batch(Ops([{}], [None], 1), np.zeros(chains, np.int32))
    b.set_csr([n] * chains, np.array(rowptr, np.int64), np.array(col, np.int32), np.array(val, complex))
    v0 = np.zeros(chains * n, complex)
    v0[::n] = 1.0
    alpha, beta, kout, _ = b.lanczos(n, reorth=1, v0=v0)
    energy, norm2 = 0.01 * rng.normal(size=chains), rng.uniform(0.5, 2.0, chains)
    sign = np.where(np.arange(chains) % 4 == 3, -1, 1)
    omega = np.linspace(-6.0, 6.0, n_w)
    args = energy, norm2, sign, np.ones(chains, np.int32), 0.02, np.zeros(chains, np.int32)
    g, spec = b.cf(*args, 1, omega, 0.1, want_g=True)
    g_many, many = b.cf(*args, 4097, omega, 0.1, want_g=True)
    assert np.array_equal(spec[0], many[0]) and not many[1:].any()
    assert np.array_equal(g, g_many)
    ref = np.zeros(n_w)
    for c in range(chains):
        a, be, k = alpha[c], beta[c], int(kout[c])
        z = sign[c] * (omega + 0.1j) + energy[c]
        f = np.zeros(n_w, complex)
        for i in range(k - 1, -1, -1):
            f = 1.0 / (z - a[i] - (be[i] ** 2 * f if i < k - 1 else 0.0))
        f *= sign[c] * norm2[c]
        assert np.abs(g[c] - f).max() <= 1e-10 * np.abs(f).max()
        ref += np.exp(-(energy[c] - energy.min()) / 0.02) * -f.imag
    ref /= np.sum(np.exp(-(energy - energy.min()) / 0.02))
    assert np.abs(spec[0] - ref).max() <= 1e-10 * max(np.abs(ref).max(), np.abs(g).max())
