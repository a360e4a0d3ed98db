"""H psi at the K lengths where the pipelined products change: no, one and
several K tiles (16, 32 rows) ahead in registers, whole and ragged, for output
sizes at the edges of 32, 64 and 128 tiles; real, complex and FP32, aligned
and unaligned rows, against the oracle's contraction; in FP64 also in place, since
small separate vectors take a one-launch product without these kernels.  Products
with K in parts, and with rows past 32-bit tile offsets."""

import ctypes as C

import numpy as np
import pytest

from oracle import tn_oracle as O
from tests.test_gpu_wstep import in_place_product

pytestmark = pytest.mark.gpu

# (chi left, chi right): the first product sums over chi left, the last over
# 3 chi right, with (3 chi left) x (4 chi right) and (4 chi left) x (chi right) outputs
SIZES = [(1, 2), (2, 11), (16, 5), (17, 31), (32, 32), (33, 43), (48, 16), (64, 64), (65, 10), (96, 3), (97, 63),
         (128, 30), (129, 65), (160, 22), (161, 86), (193, 129), (200, 140)]


@pytest.fixture(scope="module")
def T():
    import tennetlib_amd
    return tennetlib_amd


@pytest.mark.parametrize("chil,chir", SIZES)
@pytest.mark.parametrize("cplx", [False, True])
def test_products_over_k_lengths(T, chil, chir, cplx):
    rng = np.random.default_rng(chil * 1000 + chir)

    def draw(*shape):
        x = rng.standard_normal(shape)
        return x + 1j * rng.standard_normal(shape) if cplx else x

    wd, cd = [1, 3, 3, 3, 3, 1], [1, 2, chil, 5, chir, 1]
    Ws = [rng.standard_normal((wd[k], 2, 2, wd[k + 1])) for k in range(5)]
    A = [draw(cd[k], 2, cd[k + 1]) for k in range(5)]
    env, ref = T.StateEnvs(A, Ws), O.Envs(Ws, dtype=complex if cplx else float)
    cap = O.Envs([np.abs(W) for W in Ws])
    T.position_(env, 3)
    ref.position(A, 3)
    cap.position([np.abs(a) for a in A], 3)
    dims, _ = env.phi_dims()
    psi = draw(*dims)
    want = ref.product(psi)
    # rounding is bounded by eps times the contraction of the absolute values
    # times the lengths of the sums (three in the product, three in each
    # environment); |complex| products lose a factor of two at most
    scale = np.linalg.norm(cap.product(np.abs(psi))) * (2 if cplx else 1)
    n = 6 * (4 * max(chil, 2) + 3 * max(chir, 2) + 12)
    for prec, eps in (("fp64", 2.0 ** -53), ("fp32", 2.0 ** -24)):
        print("gemm", chil, chir, cplx, prec, flush=True)
        got = T.product(env, psi, precision=prec).reshape(want.shape)
        err = np.linalg.norm(got - want)
        assert err <= n * eps * scale, (prec, err / scale)
        if prec == "fp64":  # in place: three launches also where separate vectors take one
            err = np.linalg.norm(in_place_product(T, env, psi) - want)
            assert err <= n * eps * scale, ("in place", err / scale)


# K of the last product (3 chi right) split into parts of 256 (FP64) or 128 rows:
# the first split sizes, equal parts, and last parts of one row and more
@pytest.mark.parametrize("chil,chir", [(2, 85), (2, 86), (1, 128), (2, 170), (3, 171), (5, 181), (2, 256), (1, 343)])
@pytest.mark.parametrize("cplx", [False, True])
def test_products_over_split_k(T, chil, chir, cplx):
    test_products_over_k_lengths(T, chil, chir, cplx)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("p,n", [(2, 2 ** 21 + 74), (126, 2 ** 21 + 74), (2, 2 ** 22 + 74), (2, 2 ** 25 + 2)])
def test_rows_beyond_32_bit_offsets(T, p, n, cplx):
    """Products whose operands' rows are so long (n doubles) that the rows of a
    tile reach 2^31 or 2^32 bytes, those that are there or with those past the
    end: the density matrix M M^H and the other factor U^H M of a wide tensor.
    Sums of n products of a unit tensor: sqrt(n) eps in practice."""
    ctx = T.default_context()
    n = n // 4 * 2 if cplx else n
    rng = np.random.default_rng(n)
    M = rng.standard_normal((p, n))
    if cplx:
        M = M + 1j * rng.standard_normal(M.shape)
    M /= np.linalg.norm(M)
    chir = M.shape[1] // 2
    dt = M.dtype
    A = [np.ones((1, 2, p // 2), dt), np.ones((p // 2, 2, 1), dt), np.ones((1, 2, chir), dt), np.ones((chir, 2, 1), dt)]
    env = T.StateEnvs(A, T.heisenberg_mpo(4))
    dphi = T.DeviceArray.from_numpy(ctx, M.reshape(p // 2, 2, 2, chir))
    w, err, k = (C.c_double * p)(), C.c_double(), C.c_long()
    print("long rows", p, n, cplx, flush=True)
    ctx.check(ctx.lib.tn_replacebond(env.h, 2, dphi.ptr, 1, p, 1, -1.0, 0.0, 1, C.byref(err), w, p, C.byref(k)))
    a, b = env.get_site(2).reshape(p, -1), env.get_site(3).reshape(-1, M.shape[1])
    env.close()
    dphi.free()
    tol = np.sqrt(n) * 2.0 ** -52
    assert np.abs(np.array(w[:k.value]) - np.linalg.eigvalsh(M @ M.conj().T)[::-1]).max() <= tol
    assert np.linalg.norm(a @ b - M) <= tol
    assert np.abs(a.conj().T @ a - np.eye(p)).max() <= p * 1e-15


def test_block_sparse_rows_beyond_32_bit_offsets(T):
    """The QN product with an operator of 16300 channels on the right: its second
    block-sparse product reads rows of 4 * 16300 * 64 numbers.  All channels are
    diagonal, so the environment and the result are short contractions.  Sums of
    16300 * 64 products, sqrt of that in eps in practice: 1e-12 of the sums of
    absolute values."""
    rng = np.random.default_rng(5)
    w, chil, chir = 16300, 3, 64
    ql, qr = np.array([-1, -1, 1]), np.repeat([-1, 1], chir // 2)
    spin = np.array([1, -1])
    f1, f2 = rng.standard_normal(2), rng.standard_normal(2)
    f3, f4 = rng.standard_normal((2, w)), rng.standard_normal((w, 2))
    eye = np.eye(2)
    Ws = [np.einsum("ij,j->ij", eye, f)[None, :, :, None] for f in (f1, f2)]
    Ws += [np.einsum("ij,jc->ijc", eye, f3)[None], np.einsum("ij,cj->cij", eye, f4)[..., None]]
    A1 = rng.standard_normal((1, 2, chil)) * (spin[None, :, None] == ql)
    A4 = rng.standard_normal((chir, 2, 1)) * (qr[:, None, None] + spin[None, :, None] == 0)
    A2, A3 = rng.standard_normal((chil, 2, 2)), rng.standard_normal((2, 2, chir))
    env = T.StateEnvs([A1, A2, A3, A4], Ws)
    ctx, pi = env.ctx, C.POINTER(C.c_int)
    sq = np.tile(spin, 4).astype(np.int32)
    lq = np.concatenate([[0], ql, [0, 0], qr, [0]]).astype(np.int32)
    ctx.check(ctx.lib.tn_env_set_qn(env.h, 1, sq.ctypes.data_as(pi), lq.ctypes.data_as(pi)))
    T.position_(env, 2)
    mask = (ql[:, None, None, None] + spin[:, None, None] + spin[:, None] == qr)
    psi = rng.standard_normal(mask.shape) * mask

    def product(a1, a4, g1, g2, g3, g4, v):
        L = np.einsum("sa,sc,s->ac", a1[0], a1[0], g1)
        v = np.einsum("ac,cstb,s->astb", L, v, g2)
        O = g3 @ g4                                    # [spin 3, spin 4], summed over the channels
        R = np.einsum("bs,cs,ts->tbc", a4[..., 0], a4[..., 0], O)
        return np.einsum("astb,tbc->astc", v, R)

    print("long block rows", flush=True)
    got = T.product(env, psi).reshape(psi.shape)
    want = product(A1, A4, f1, f2, f3, f4, psi) * mask
    cap = product(*(np.abs(x) for x in (A1, A4, f1, f2, f3, f4, psi)))
    assert np.linalg.norm(got - want) <= 1e-12 * np.linalg.norm(cap)
    env.close()
