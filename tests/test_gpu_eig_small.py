"""Factorisations at the sizes where the density-matrix eigensolver changes
kernels: blocks of one workgroup (tridiagonalisation classes 32, 64, 128 and
192 rows, divide and conquer classes 32, 64, 128), the first sizes above them
(leaves and merges, the last columns by one workgroup) and the register limits
of the back-transformation (real 768, complex 384).

Compared with the factors that the matrix is built from: weights to a few
rounding errors of the largest one, the product of the two factors with the
matrix, and the kept factor's orthonormality (each sum of n products of unit
vectors rounds to about n / 2 eps at the worst, sqrt(n) eps in practice)."""

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.fixture(scope="module")
def T():
    import tennetlib_amd
    return tennetlib_amd


def spectra(n, kind):
    i = np.arange(n)
    if kind == "graded":          # weights far below rounding of the largest
        s = 10.0 ** (-9.0 * i / n)
    elif kind == "multiplets":    # degenerate triples: Givens deflation
        s = 10.0 ** (-np.floor(i / 3) / 8.0)
    else:                         # half the weights exactly zero
        s = np.where(i < (n + 1) // 2, 1.0 / (1.0 + i), 0.0)
    return s / np.linalg.norm(s)


def factorise(T, phi, left):
    chil, d, _, chir = phi.shape
    ctx = T.default_context()
    dt = phi.dtype
    A = [np.ones((1, d, chil), dt), np.ones((chil, d, 1), dt), np.ones((1, d, chir), dt), np.ones((chir, d, 1), dt)]
    env = T.StateEnvs(A, T.heisenberg_mpo(4))
    m, n = chil * d, chir * d
    dphi = T.DeviceArray.from_numpy(ctx, phi)
    w, err, k = (C.c_double * (m + n))(), C.c_double(), C.c_long()
    ctx.check(ctx.lib.tn_replacebond(env.h, 2, dphi.ptr, int(left), m + n, 1, -1.0, 0.0, 1, C.byref(err), w, m + n,
                                     C.byref(k)))
    a, b = env.get_site(2), env.get_site(3)
    env.close()
    return a, b, np.array(w[:k.value])


@pytest.mark.parametrize("kind", ["graded", "multiplets", "rank"])
@pytest.mark.parametrize("cplx,chi", [(False, c) for c in (1, 2, 15, 16, 17, 32, 33, 63, 64, 65, 96, 97, 128, 129,
                                                           191, 257, 384, 385)] +
                         [(True, c) for c in (1, 2, 15, 16, 17, 32, 33, 63, 64, 65, 96, 97, 128, 192, 193)])
def test_factorisation_at_eigensolver_size_classes(T, kind, cplx, chi):
    rng = np.random.default_rng(chi + 1000 * cplx)
    p = 2 * chi

    def unitary():
        a = rng.standard_normal((p, p))
        if cplx:
            a = a + 1j * rng.standard_normal((p, p))
        return np.linalg.qr(a)[0]

    s = spectra(p, kind)
    M = (unitary() * s) @ unitary().conj().T
    phi = np.ascontiguousarray(M.reshape(chi, 2, 2, chi)).astype(np.complex128 if cplx else np.float64)
    for left in (True, False):
        a, b, w = factorise(T, phi, left)
        k = len(w)
        assert np.abs(np.sort(w)[::-1] - np.sort(s ** 2)[::-1][:k]).max() <= 40 * EPS
        A, B = a.reshape(p, k), b.reshape(k, p)
        assert np.abs(A @ B - M).max() <= 40 * EPS
        Q = A if left else B.conj().T
        assert np.abs(Q.conj().T @ Q - np.eye(k)).max() <= 60 * EPS


def test_factorisation_extreme_scales(T):
    """A tensor scaled by a large power of two has the same factors and weights
    scaled exactly: the reduction and the divide and conquer of up to 128 rows
    work on scaled entries (the exponents of larger ones, whose column kernels
    sum squares of the density matrix: 4 |e| below 1022 less the 40 bits of its
    entries; those of small ones are below)."""
    rng = np.random.default_rng(3)
    phi = rng.standard_normal((20, 2, 2, 20))
    phi /= np.linalg.norm(phi)
    ref = factorise(T, phi, True)
    for e in (-220, 220):
        a, b, w = factorise(T, np.ldexp(phi, e), True)
        assert np.abs(np.ldexp(w, -2 * e) - ref[2]).max() <= 40 * EPS
        assert np.abs(a.reshape(40, -1) @ b.reshape(-1, 40) - phi.reshape(40, 40)).max() <= 40 * EPS


@pytest.mark.parametrize("chi", [2, 3, 10, 50])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("e", [-515, -400, -270, -267, -262])
@pytest.mark.parametrize("tiny_first", [False, True])
def test_factorisation_of_blocks_of_unlike_scale(T, chi, cplx, e, tiny_first):
    """A dense block of the density matrix at 2^(2e) beside one at one (its
    entries or their products below the normal range): the factors of the block
    at one to its rounding, and all vectors orthonormal."""
    rng = np.random.default_rng(chi)
    p = 2 * chi
    M = np.zeros((p, p), np.complex128 if cplx else np.float64)
    for rows, scale in ((slice(0, chi), 0 if not tiny_first else e), (slice(chi, p), e if not tiny_first else 0)):
        b = rng.standard_normal((chi, chi))
        if cplx:
            b = b + 1j * rng.standard_normal((chi, chi))
        M[rows, rows] = b / np.linalg.norm(b) * 2.0 ** scale
    print("unlike", chi, cplx, e, tiny_first, flush=True)
    for left in (True, False):
        a, b, w = factorise(T, np.ascontiguousarray(M.reshape(chi, 2, 2, chi)), left)
        k = len(w)
        want = np.sort(np.linalg.svd(M, compute_uv=False) ** 2)[::-1][:k]
        assert np.abs(np.sort(w)[::-1] - want).max() <= 40 * EPS
        A, B = a.reshape(p, k), b.reshape(k, p)
        assert np.abs(A @ B - M).max() <= 40 * EPS
        Q = A if left else B.conj().T
        assert np.abs(Q.conj().T @ Q - np.eye(k)).max() <= 60 * EPS


@pytest.mark.parametrize("chi,cplx", [(1, False), (2, False), (4, False), (7, True), (20, False), (50, True),
                                      (64, True), (64, False)])
@pytest.mark.parametrize("e", [-480, -400, 400, 500])
def test_small_factorisation_scales_exactly(T, chi, cplx, e):
    """Factorisations of up to 128 rows (one workgroup a stage) of a
    unit tensor times 2^e: the same factors (the new sites are normalised), the
    weights times 2^(2e), which stay normal numbers while their squares do not."""
    rng = np.random.default_rng(chi)
    phi = rng.standard_normal((chi, 2, 2, chi))
    if cplx:
        phi = phi + 1j * rng.standard_normal((chi, 2, 2, chi))
    phi /= np.linalg.norm(phi)
    ref = factorise(T, phi, True)
    print("scaled", chi, cplx, e, flush=True)
    a, b, w = factorise(T, phi * 2.0 ** e, True)
    p = 2 * chi
    # entries of the density matrix under 2^-1022 keep an absolute error of 2^-1075
    assert np.abs(np.ldexp(w, -2 * e) - ref[2]).max() <= 40 * EPS
    A, B = a.reshape(p, -1), b.reshape(-1, p)
    assert np.abs(A @ B - phi.reshape(p, p)).max() <= 40 * EPS
    assert np.abs(A.conj().T @ A - np.eye(A.shape[1])).max() <= 60 * EPS
