"""The estimate that decides the grid-wide eigensolver's Gram-Schmidt passes (csrc/orth_estimate.h,
plain C++, built here with the host compiler) on Lanczos runs in numpy.

The rule keeps |<v_j, v_k>| at kOrthLevel = 1e-13 or, where less, 8 eps |H| / |H - sigma|: a pass comes
before the estimate exceeds it, so the true products may exceed it by what the estimate misses in one
step; 10 times the level is allowed.  (Below 1e-14 every step passes.)  Far from zero energy (|H| / |H - sigma| over 50) the passes must
be the exception, in fewer than half of the steps.
"""

import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest
import scipy.sparse

LEVEL = 1e-13
CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "impuritymodel_amd", "csrc")


@pytest.fixture(scope="module")
def estimate(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("orth")
    (d / "e.cpp").write_text(
        '#include "orth_estimate.h"\n'
        "using imped::OrthEstimate;\n"
        'extern "C" {\n'
        "void* make(double sigma) { return new OrthEstimate(sigma); }\n"
        "void drop(void* e) { delete (OrthEstimate*)e; }\n"
        "int step(void* e, double al, double bt) { return ((OrthEstimate*)e)->step(al, bt); }\n"
        "void done(void* e, double bt, int passed) { ((OrthEstimate*)e)->done(bt, passed != 0); }\n"
        "}\n")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I" + CSRC, str(d / "e.cpp"), "-o", str(d / "e.so")],
                   check=True)
    lib = ctypes.CDLL(str(d / "e.so"))
    lib.make.restype = ctypes.c_void_p
    lib.make.argtypes = [ctypes.c_double]
    lib.drop.argtypes = [ctypes.c_void_p]
    lib.step.argtypes = [ctypes.c_void_p, ctypes.c_double, ctypes.c_double]
    lib.done.argtypes = [ctypes.c_void_p, ctypes.c_double, ctypes.c_int]
    return lib


def _matrix(n, width, shift, complex_h):
    rng = np.random.default_rng(n)

    def part():
        return scipy.sparse.random(n, n, density=6.0 / n, random_state=rng,
                                   data_rvs=lambda k: width * rng.standard_normal(k)).toarray()

    a = part() + (1j * part() if complex_h else 0.0)
    return a + a.conj().T + np.diag(2 * width * rng.standard_normal(n) + shift)


def _run(lib, h, shifted, steps):
    """(passes, largest |<v_j, v_k>|) of a Lanczos run with the estimate's passes."""
    rng = np.random.default_rng(0)
    v = rng.standard_normal(len(h)).astype(h.dtype)
    V = [v / np.linalg.norm(v)]
    sigma = np.vdot(V[0], h @ V[0]).real if shifted else 0.0
    h = h - sigma * np.eye(len(h))
    hs = scipy.sparse.csr_matrix(h)
    e, beta, passes = lib.make(sigma), [], 0
    for j in range(steps):
        w = hs @ V[-1]
        al = np.vdot(V[-1], w).real
        w = w - al * V[-1] - (beta[-1] * V[-2] if j else 0.0)
        b = np.linalg.norm(w)
        passed = lib.step(e, al, b)
        if passed:
            passes += 1
            m = np.array(V)
            w = w - m.T @ (m.conj() @ w)
            if np.linalg.norm(w) ** 2 < 0.5 * b ** 2:
                w = w - m.T @ (m.conj() @ w)
            b = np.linalg.norm(w)
        lib.done(e, b, passed)
        beta.append(b)
        V.append(w / b)
    lib.drop(e)
    g = np.array(V).conj() @ np.array(V).T
    np.fill_diagonal(g, 0.0)
    return passes, np.abs(g).max()


@pytest.mark.parametrize("n,width,shift,complex_h", [(700, 1.0, -900.0, False), (500, 1.0, -900.0, True),
                                                     (600, 0.2, -900.0, False), (600, 0.02, 300.0, True)])
def test_passes_are_few_and_keep_the_level(estimate, n, width, shift, complex_h):
    passes, worst = _run(estimate, _matrix(n, width, shift, complex_h), True, 140)
    assert 0 < passes < 70
    assert worst <= 10 * LEVEL


@pytest.mark.parametrize("complex_h", [False, True])
def test_near_zero_energy_every_step_passes(estimate, complex_h):
    # |H| = |H - sigma|: 8 to 16 eps is no level to save passes at
    passes, worst = _run(estimate, _matrix(400, 1.0, 0.0, complex_h), True, 140)
    assert passes == 140
    assert worst <= 1e-14


def test_energies_far_from_zero_need_the_shift(estimate):
    # |alpha| eps over the hopping alone passes the level: every step makes its pass
    assert _run(estimate, _matrix(600, 0.02, -900.0, False), False, 60)[0] == 60
