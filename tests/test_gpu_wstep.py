"""H psi where the operator step changes kernels: operators of one to 128 rows
and columns (blocks of 16 rows in FP64, 32 in FP32, K groups of 20 and 10),
dense and sparse, with column counts at the edges of a strip (32 and 64), odd
ones and one column, against the oracle's contraction; in FP64 also in place,
since small separate vectors take a one-launch product without this step."""

import numpy as np
import pytest

from oracle import tn_oracle as O

pytestmark = pytest.mark.gpu

# (MPO bond, d, sites, chi left, chi right): rows and columns = bond * d^sites
SIZES = [(1, 2, 1, 5, 1), (5, 2, 1, 16, 33), (8, 2, 1, 16, 64), (17, 1, 1, 9, 31), (5, 2, 2, 40, 64),
         (8, 2, 2, 3, 66), (11, 3, 1, 7, 65), (4, 4, 2, 16, 30), (20, 2, 2, 33, 97), (24, 2, 2, 20, 32),
         (7, 4, 2, 6, 34), (32, 2, 2, 37, 63), (8, 4, 2, 64, 128), (24, 2, 1, 64, 65), (16, 2, 2, 33, 98),
         (20, 2, 2, 17, 66), (24, 2, 2, 64, 65), (6, 4, 2, 64, 66), (7, 4, 2, 33, 67), (3, 2, 1, 40, 1)]


@pytest.fixture(scope="module")
def T():
    import tennetlib_amd
    return tennetlib_amd


def chain(w, d, chil, chir, fill, seed):
    """Four sites with a random MPO of bond w around sites 2 and 3."""
    rng = np.random.default_rng(seed)
    wd = [1, w, w, w, 1]
    cd = [1, min(chil, 8), chil, chir, 1]
    Ws = []
    for k in range(4):
        W = rng.standard_normal((wd[k], d, d, wd[k + 1]))
        Ws.append(W * (rng.random(W.shape) < fill))
    A = [rng.standard_normal((cd[k], d, cd[k + 1])) for k in range(4)]
    return Ws, A, rng


def in_place_product(T, env, psi):
    """H psi in FP64 with the output over the input, which takes the GEMM, the
    operator step and the GEMM at any size."""
    buf = T.DeviceArray.from_numpy(env.ctx, psi)
    env.ctx.check(env.ctx.lib.tn_env_matvec(env.h, buf.ptr, buf.ptr, 0))
    out = buf.numpy()
    buf.free()
    return out


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "w%d_d%d_n%d_%dx%d" % s)
@pytest.mark.parametrize("fill", [1.0, 0.15])
def test_operator_step(T, size, fill):
    w, d, nsite, chil, chir = size
    Ws, A, rng = chain(w, d, chil, chir, fill, seed=w * 1000 + chir)
    env, ref = T.StateEnvs(A, Ws), O.Envs(Ws)
    ref.nsite = nsite
    T.set_nsite_(env, nsite)
    p = 2 if nsite == 2 else 3   # one site: both of its bonds are chil and chir wide
    T.position_(env, p)
    ref.position(A, p)
    dims, _ = env.phi_dims()
    psi = rng.standard_normal(tuple(dims) if nsite == 2 else (dims[0], dims[1], dims[3]))
    want = ref.product(psi)
    # rounding grows with the lengths of the sums and with the cancellation in
    # them: bounded by eps times the product of the absolute values, whose norm
    # is taken from the same contraction
    cap = O.Envs([np.abs(W) for W in Ws])
    cap.nsite = nsite
    cap.position([np.abs(a) for a in A], p)
    scale = np.linalg.norm(cap.product(np.abs(psi)))
    # relative error of one sum of K products: K eps at the worst, sqrt(K) in
    # practice; three sums of at most 4 * 128 terms follow each other in the
    # environments and three in the product, and the precision's own input
    # rounding (2^-24; bf16 pairs 2^-16, kept to 1e-4 elsewhere) is inside
    for prec, tol in (("fp64", 6 * 512 * 2.0 ** -53), ("fp32", 3 * 512 * 2.0 ** -24), ("bf16x3", 1e-4)):
        print("w step", size, fill, prec, flush=True)
        got = T.product(env, psi, precision=prec).reshape(want.shape)
        err = np.linalg.norm(got - want)
        assert err <= tol * scale, (prec, err / max(scale, 1e-300))
        if prec == "fp64":  # in place: three launches also where separate vectors take one
            err = np.linalg.norm(in_place_product(T, env, psi) - want)
            assert err <= tol * scale, ("in place", err / max(scale, 1e-300))


@pytest.mark.parametrize("chi", [8, 15, 64, 65])
@pytest.mark.parametrize("cplx,prec", [(False, "fp64"), (False, "fp32"), (False, "bf16x3"), (True, "fp64"),
                                       (True, "fp32")])
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_operator_zeros_leave_non_finite_values_out(T, chi, cplx, prec, value):
    """An Inf or NaN in psi at the spins (up, up) reaches only the rows that the
    operator couples to them: a Heisenberg bond does not flip both spins, so
    the rows (down, down) are those of psi with a zero in its place.  One launch
    (chi = 8, 15 in FP64) and three, even and odd column counts.  Tolerance as
    for the products above: other sums, of at most 5 chi terms."""
    rng = np.random.default_rng(chi + cplx)

    def draw(*shape):
        x = rng.standard_normal(shape)
        return x + 1j * rng.standard_normal(shape) if cplx else x

    cd = [1, 2, chi, 4, chi, 2, 1]
    A = [draw(cd[k], 2, cd[k + 1]) / np.sqrt(cd[k] * cd[k + 1]) for k in range(6)]
    env = T.StateEnvs(A, O.heisenberg_mpo(6))
    T.position_(env, 3)
    dims, _ = env.phi_dims()
    psi = draw(*dims)
    psi[chi // 2, 0, 0, chi // 3] = 0.0
    want = T.product(env, psi, precision=prec).reshape(dims)[:, 1, 1]
    psi[chi // 2, 0, 0, chi // 3] = value
    print("zeros", chi, cplx, prec, value, flush=True)
    got = T.product(env, psi, precision=prec).reshape(dims)
    assert not np.isfinite(got[:, 0, 0]).any()
    eps = 2.0 ** -53 if prec == "fp64" else 2.0 ** -24
    assert np.linalg.norm(got[:, 1, 1] - want) <= 15 * chi * eps * np.linalg.norm(want)
