"""H psi of small bonds in one launch: odd and even sizes around the tiles (16),
the workgroups' share of the left bond, split and unsplit sums of the last
product, up to the sizes that take three launches instead, one and two sites,
real and complex, dense and sparse operators, on host-called, allocation-free
and repeated products, against the oracle's contraction."""

import numpy as np
import pytest

from oracle import tn_oracle as O

pytestmark = pytest.mark.gpu

# (MPO bonds left and right of the pair, d, sites, chi left, chi right)
SIZES = [(1, 1, 1, 1, 1, 1), (1, 1, 2, 1, 3, 2), (2, 3, 2, 1, 5, 7), (5, 5, 2, 2, 1, 16), (5, 5, 2, 2, 16, 1),
         (5, 4, 2, 2, 15, 17), (5, 5, 2, 2, 16, 16), (5, 5, 2, 2, 31, 33), (5, 5, 2, 2, 33, 31), (3, 7, 3, 1, 20, 22),
         (6, 6, 4, 2, 9, 14), (8, 8, 4, 2, 6, 11), (17, 3, 2, 2, 10, 19), (20, 20, 2, 2, 18, 21), (32, 32, 2, 2, 4, 9),
         (5, 5, 2, 1, 50, 20), (5, 5, 2, 2, 2, 60), (5, 5, 2, 2, 60, 2), (1, 1, 2, 2, 49, 48), (2, 2, 3, 2, 40, 41)]


@pytest.fixture(scope="module")
def T():
    import tennetlib_amd
    return tennetlib_amd


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "w%d_%d_d%d_n%d_%dx%d" % s)
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("fill", [1.0, 0.2])
def test_one_launch_product(T, size, cplx, fill):
    wl, wr, d, nsite, chil, chir = size
    rng = np.random.default_rng(sum(size) + 10 * cplx)

    def draw(*shape):
        x = rng.standard_normal(shape)
        return x + 1j * rng.standard_normal(shape) if cplx else x

    # the bonds of the position in the middle: sites p and p + 1, or site p
    wd = [1, wl, wr, 1] if nsite == 1 else [1, wl, 3, wr, 1]
    cd = [1, chil, chir, 1] if nsite == 1 else [1, chil, 3, chir, 1]
    N = len(wd) - 1
    Ws = []
    for k in range(N):
        W = rng.standard_normal((wd[k], d, d, wd[k + 1]))
        Ws.append(W * (rng.random(W.shape) < fill))
    A = [draw(cd[k], d, cd[k + 1]) for k in range(N)]
    env, ref = T.StateEnvs(A, Ws), O.Envs(Ws, dtype=complex if cplx else float)
    cap = O.Envs([np.abs(W) for W in Ws])
    ref.nsite = cap.nsite = nsite
    T.set_nsite_(env, nsite)
    T.position_(env, 2)
    ref.position(A, 2)
    cap.position([np.abs(a) for a in A], 2)
    dims, n = env.phi_dims()
    psi = draw(*(dims if nsite == 2 else (dims[0], dims[1], dims[3])))
    want = ref.product(psi)
    # eps per term of every sum (three in the product, three in each
    # environment) of the contraction of absolute values; a factor of two for
    # complex products
    terms = 3 * 3 * max(chil, chir * wr, wl * d * d, 16)
    scale = np.linalg.norm(cap.product(np.abs(psi))) * (2 if cplx else 1)
    print("mv", size, cplx, fill, flush=True)
    got = T.product(env, psi).reshape(want.shape)
    assert np.linalg.norm(got - want) <= terms * 2.0 ** -53 * scale
    # the allocation-free entry and a repeated call take the same path
    dv, out = T.DeviceArray.from_numpy(env.ctx, psi), T.DeviceArray(env.ctx, psi.shape, env.dtype)
    env.ctx.check(env.ctx.lib.tn_env_matvec_noalloc(env.h, dv.ptr, out.ptr))
    assert np.array_equal(out.numpy().reshape(-1), got.reshape(-1))
    assert np.array_equal(T.product(env, psi).reshape(-1), got.reshape(-1))
    dv.free()
    out.free()


@pytest.mark.parametrize("chi", [16, 64])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("noalloc", [False, True])
def test_product_in_place(T, chi, cplx, noalloc):
    """out == v, and out overlapping the end of v: the separate product's
    result.  chi = 16 takes one launch with separate vectors, 64 three.  Other
    kernels sum in another order: eps per term of the sums as above, on
    vectors of norm |psi| |H|."""
    rng = np.random.default_rng(chi + cplx)

    def draw(*shape):
        x = rng.standard_normal(shape)
        return x + 1j * rng.standard_normal(shape) if cplx else x

    cd = [1, 2, chi, 4, chi, 2, 1]
    A = [draw(cd[k], 2, cd[k + 1]) / np.sqrt(cd[k] * cd[k + 1]) for k in range(6)]
    env = T.StateEnvs(A, O.heisenberg_mpo(6))
    T.position_(env, 3)
    dims, n = env.phi_dims()
    psi = draw(*dims).reshape(-1)
    want = T.product(env, psi.reshape(dims)).reshape(-1)
    tol = 3 * 5 * chi * 2.0 ** -53 * np.linalg.norm(np.abs(want)) * (2 if cplx else 1)
    item = np.dtype(env.dtype).itemsize
    for shift in (0, n - 3):
        buf = T.DeviceArray.from_numpy(env.ctx, np.concatenate([psi, np.zeros_like(psi)]).astype(env.dtype))
        v, out = buf.ptr.value, buf.ptr.value + shift * item
        print("in place", chi, cplx, noalloc, shift, flush=True)
        if noalloc:
            env.ctx.check(env.ctx.lib.tn_env_matvec_noalloc(env.h, v, out))
        else:
            env.ctx.check(env.ctx.lib.tn_env_matvec(env.h, v, out, 0))
        got = buf.numpy()[shift:shift + n]
        buf.free()
        assert np.linalg.norm(got - want) <= tol
