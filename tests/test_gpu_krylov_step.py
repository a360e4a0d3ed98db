"""Lanczos solves at the vector lengths and basis sizes where a step changes
kernels: one workgroup with one element a thread (up to 1024), four (up to
4096), a launch per pass above; bases of up to 4, 8 and 16 vectors and more;
real and complex; vectors shorter than the basis, against the oracle's solver.

The Ritz value is that of an exactly orthonormal basis up to the rounding of the
kdim products, kdim eps |H| each with cancellation in sums of up to 10^4 terms:
1e-12 |H|.  Vectors agree to that over the gap of the projected matrix: 1e-8.
exp(tH) x converges to its own tolerance."""

import ctypes as C

import numpy as np
import pytest

from oracle import tn_oracle as O

pytestmark = pytest.mark.gpu

# (chi left, chi right): 4 chi left * chi right elements
SIZES = [(1, 1), (2, 3), (4, 4), (5, 13), (16, 16), (19, 27), (32, 32), (33, 32), (37, 61)]


@pytest.fixture(scope="module")
def T():
    import tennetlib_amd
    return tennetlib_amd


def setup(T, chil, chir, cplx):
    rng = np.random.default_rng(chil * 100 + chir)

    def draw(*shape):
        x = rng.standard_normal(shape)
        return x + 1j * rng.standard_normal(shape) if cplx else x

    Ws = O.xxz_mpo(6, 1.0, 0.7, np.linspace(-0.4, 0.6, 6))
    cd = [1, 2, chil, 3, chir, 2, 1]
    A = [draw(cd[k], 2, cd[k + 1]) / np.sqrt(cd[k] * cd[k + 1]) for k in range(6)]
    env, ref = T.StateEnvs(A, Ws), O.Envs(Ws, dtype=complex if cplx else float)
    T.position_(env, 3)
    ref.position(A, 3)
    dims, n = env.phi_dims()
    x = draw(*dims)
    return env, ref, x


@pytest.mark.parametrize("chil,chir", SIZES)
@pytest.mark.parametrize("cplx", [False, True])
def test_eig(T, chil, chir, cplx):
    env, ref, x = setup(T, chil, chir, cplx)
    ctx = env.ctx
    scale = np.linalg.norm(ref.product(x)) / np.linalg.norm(x)
    for kd in (2, 4, 5, 9, 16, 18, 34):
        if kd >= x.size:
            continue
        print("eig", chil, chir, cplx, kd, flush=True)
        th_ref, y_ref, info_ref = O.eigsolve_lanczos(ref.product, x, krylovdim=kd, maxiter=1, tol=1e-14)
        scale = max(scale, abs(th_ref))
        dx = T.DeviceArray.from_numpy(ctx, x)
        th, info = C.c_double(), T._lib.KrylovInfo()
        ctx.check(ctx.lib.tn_krylov_eig(env.h, dx.ptr, kd, 1, 1e-14, 0, C.byref(th), C.byref(info)))
        y = dx.numpy()
        dx.free()
        assert abs(th.value - th_ref) <= 1e-12 * scale
        assert abs(np.linalg.norm(y) - 1.0) <= 1e-14 * np.sqrt(kd)
        # the value is the vector's own, and the vector the oracle's
        assert abs(np.vdot(y, ref.product(y)).real - th.value) <= 1e-12 * scale
        assert abs(abs(np.vdot(y, y_ref)) - 1.0) <= 1e-8


@pytest.mark.parametrize("chil,chir", SIZES)
@pytest.mark.parametrize("cplx", [False, True])
def test_expm(T, chil, chir, cplx):
    env, ref, x = setup(T, chil, chir, cplx)
    ctx = env.ctx
    scale = np.linalg.norm(ref.product(x)) / np.linalg.norm(x)
    t = (0.3 - 0.4j if cplx else -0.5) / scale
    want, _ = O.exponentiate_lanczos(ref.product, t, x, krylovdim=30, maxiter=100, tol=1e-12)
    dx = T.DeviceArray.from_numpy(ctx, x)
    info = T._lib.KrylovInfo()
    print("expm", chil, chir, cplx, flush=True)
    ctx.check(ctx.lib.tn_krylov_expm(env.h, dx.ptr, np.real(t), np.imag(t), 30, 100, 1e-12, 0, C.byref(info)))
    y = dx.numpy()
    dx.free()
    assert info.converged == 1
    assert np.linalg.norm(y - want) <= 2.5e-12 * max(1.0, np.linalg.norm(want))


@pytest.mark.parametrize("chil,chir", [(128, 128), (128, 129), (300, 437)])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("kd", [3, 7, 18])
def test_eig_of_long_vectors(T, chil, chir, cplx, kd):
    """The last size whose passes sum the previous launch's 128 partial results
    themselves and the first that has them summed by a launch, and 1025 tiles of
    512 elements for the 1024 workgroups: the value and vector against the
    oracle's, and the value against the vector's own."""
    env, ref, x = setup(T, chil, chir, cplx)
    ctx = env.ctx
    print("long eig", chil, chir, cplx, kd, flush=True)
    th_ref, y_ref, _ = O.eigsolve_lanczos(ref.product, x, krylovdim=kd, maxiter=1, tol=1e-14)
    dx = T.DeviceArray.from_numpy(ctx, x)
    th, info = C.c_double(), T._lib.KrylovInfo()
    ctx.check(ctx.lib.tn_krylov_eig(env.h, dx.ptr, kd, 1, 1e-14, 0, C.byref(th), C.byref(info)))
    y = dx.numpy()
    dx.free()
    scale = max(np.linalg.norm(ref.product(x)) / np.linalg.norm(x), abs(th_ref))
    assert abs(th.value - th_ref) <= 1e-12 * scale
    assert abs(np.linalg.norm(y) - 1.0) <= 1e-14 * np.sqrt(kd)
    assert abs(np.vdot(y, ref.product(y)).real - th.value) <= 1e-12 * scale
    assert abs(abs(np.vdot(y, y_ref)) - 1.0) <= 1e-8


def test_zero_start_vectors(T):
    env, _, x = setup(T, 16, 16, False)
    ctx = env.ctx
    dx = T.DeviceArray.from_numpy(ctx, 0 * x)
    th, info = C.c_double(), T._lib.KrylovInfo()
    with pytest.raises(Exception, match="zero or non-finite start vector"):
        ctx.check(ctx.lib.tn_krylov_eig(env.h, dx.ptr, 4, 1, 1e-14, 0, C.byref(th), C.byref(info)))
    ctx.check(ctx.lib.tn_krylov_expm(env.h, dx.ptr, -0.5, 0.0, 30, 100, 1e-12, 0, C.byref(info)))
    assert not np.any(dx.numpy())
    dx.free()
