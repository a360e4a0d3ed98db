"""Factorisations of density matrices whose tridiagonalisation changes kernels:
the first sizes with columns beyond the last 192 (real), rows that fill one,
four, eight or sixteen registers of a wavefront (256, 512, 1020 entries) and the
first beyond, and the panels of 32 columns (from 3072 rows) with whole and
ragged chunks of 64 entries, up to more than 64 of them.

Compared as in test_gpu_eig_small, with p eps / 4 for the roundings of the p
reflectors that every vector passes (p eps at the worst)."""

import numpy as np
import pytest

from tests.test_gpu_eig_small import EPS, T, factorise, spectra  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,p", [(k, p) for p in (194, 196, 258, 260, 450, 514, 516, 770)
                                    for k in ("graded", "multiplets", "rank")] +
                         [("graded", 1020), ("rank", 1022), ("multiplets", 1024), ("graded", 1218), ("rank", 3070),
                          ("graded", 3072), ("multiplets", 3074), ("graded", 4162)])
def test_factorisation_at_column_kernels(T, kind, p):  # noqa: F811
    rng = np.random.default_rng(p)

    def unitary(n):
        return np.linalg.qr(rng.standard_normal((p, n)))[0]

    n = p if p < 2000 else 400  # large ones: 400 weights, the rest zero
    s = spectra(n, kind)
    print("columns", kind, p, flush=True)
    M = (unitary(n) * s) @ unitary(n).T
    phi = np.ascontiguousarray(M.reshape(p // 2, 2, 2, p // 2))
    tol = p * EPS / 4
    for left in ((True, False) if p < 1000 else (p % 4 == 2,)):
        a, b, w = factorise(T, phi, left)
        k = len(w)
        want = np.zeros(k)
        want[:min(k, n)] = np.sort(s ** 2)[::-1][:k]
        assert np.abs(np.sort(w)[::-1] - want).max() <= tol
        A, B = a.reshape(p, k), b.reshape(k, p)
        assert np.abs(A @ B - M).max() <= tol
        Q = A if left else B.T
        assert np.abs(Q.T @ Q - np.eye(k)).max() <= tol
