"""H psi at the K lengths where the pipelined products change: no, one and
several K tiles (16, 32 rows) ahead in registers, whole and ragged, for output
sizes at the edges of 32, 64 and 128 tiles; real, complex and FP32, aligned
and unaligned rows, against the oracle's contraction."""

import numpy as np
import pytest

from oracle import tn_oracle as O

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
