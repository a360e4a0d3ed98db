"""QN-conserving factorisation with sectors at the sizes where the batched
eigensolver changes: one row, one workgroup (128 rows), two leaves of the
divide and conquer, the last columns by one workgroup (192), the register
classes of the back-transformation (256, 512, 768) and the first size beyond
the batch, all in one call and alone with small ones, full rank and rank
deficient, against numpy's eigenvectors block by block.

Weights of a unit tensor: a few roundings of the largest one, 1e-13.  Kept
vectors orthonormal to sums of n <= 769 products of unit vectors (sqrt(n) eps
each, 1e-13); the product of the two new sites loses what is cut, and sums of
as many products, 1e-12."""

import ctypes as C

import numpy as np
import pytest

from oracle import tn_oracle as O
from oracle import tn_oracle_qn as Q

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    import tennetlib_amd
    return tennetlib_amd


def left_sizes(sectors):
    """Link sizes whose neighbours' sums are the wanted sectors of (link, spin 1/2)."""
    a = [sectors[0]]
    for p in sectors[1:]:
        a.append(p - a[-1])
    assert min(a) > 0
    return a


CASES = {
    "one": ([1], 3),
    "small": ([2, 3, 32, 33, 64, 65, 127, 128], 40),
    "edges": ([1, 128, 129, 192, 193], 150),
    "deficient": ([5, 129, 193, 256, 257, 300], 20),
    "all": ([1, 128, 129, 192, 193, 256, 257, 512, 513, 768, 769], 30),
}


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("ortho", ["left", "right"])
def test_sector_sizes(T, case, ortho):
    run_case(T, case, ortho)


@pytest.mark.parametrize("ortho", ["left", "right"])
@pytest.mark.parametrize("e", [-400, 400])
def test_sector_scales(T, ortho, e):
    """The unit tensor times 2^e: the same vectors (the new sites are
    normalised), the weights times 2^(2e)."""
    run_case(T, "small", ortho, e)


def run_case(T, case, ortho, e=0):
    sectors, chir = CASES[case]
    sizes = left_sizes(sectors)
    qs = Q.spin_half_qns()
    ql = [(2 * i,) for i, n in enumerate(sizes) for _ in range(n)]
    qr = [(2 * i,) for i in range(-2, len(sizes) + 2) for _ in range(chir)]
    if ortho == "right":
        # the mirror image: the sectors of (spin 1/2, right link)
        ql, qr = [(-q[0],) for q in qr], [(-q[0],) for q in ql]
    rng = np.random.default_rng(len(ql) + len(qr))
    fl = np.add.outer(np.add.outer(np.array([q[0] for q in ql]), np.array([q[0] for q in qs])),
                      np.array([q[0] for q in qs]))
    mask = fl[..., None] == np.array([q[0] for q in qr])
    phi = rng.standard_normal(mask.shape) * mask
    phi *= np.exp(-4.0 * np.arange(len(ql)) / len(ql))[:, None, None, None]
    phi /= np.linalg.norm(phi)
    N, b, chim = 4, 2, 8
    dims = [1, len(ql), chim, len(qr), 1]
    A = [rng.standard_normal((dims[k], 2, dims[k + 1])) for k in range(N)]
    env = T.StateEnvs(A, O.heisenberg_mpo(N))
    ctx = env.ctx
    pi = C.POINTER(C.c_int)
    sq = np.array([x for _ in range(N) for q in qs for x in q], dtype=np.int32)
    lq = np.array([x for lk in [[(0,)], ql, [(0,)] * chim, qr, [(0,)]] for q in lk for x in q], dtype=np.int32)
    ctx.check(ctx.lib.tn_env_set_qn(env.h, 1, sq.ctypes.data_as(pi), lq.ctypes.data_as(pi)))
    env.nq = 1
    Ab, Ab1, newq, spec = Q.block_factorize(phi, ql, qs, qs, qr, 10 ** 6, 1, 1e-13, ortho)
    dphi = T.DeviceArray.from_numpy(ctx, phi * 2.0 ** e)
    terr, nk = C.c_double(), C.c_long()
    eigs = (C.c_double * 8192)()
    print("qn blocks", case, ortho, e, flush=True)
    ctx.check(ctx.lib.tn_replacebond(env.h, b, dphi.ptr, 1 if ortho == "left" else 0, 10 ** 6, 1, 1e-13, 0.0, 1,
                                     C.byref(terr), eigs, 8192, C.byref(nk)))
    assert nk.value == len(newq)
    assert np.abs(np.ldexp(np.array(eigs[:nk.value]), -2 * e) - spec.eigs).max() < 1e-13
    assert env.sectors(b) == spec.sectors
    got = [env.get_site(b), env.get_site(b + 1)]
    U = got[0].reshape(-1, nk.value) if ortho == "left" else got[1].reshape(nk.value, -1).T
    assert np.abs(U.T @ U - np.eye(nk.value)).max() < 1e-13
    m = got[0].shape[0] * 2
    prod = got[0].reshape(m, -1) @ got[1].reshape(nk.value, -1)
    want = Ab.reshape(m, -1) @ Ab1.reshape(nk.value, -1)
    assert np.abs(prod - want).max() < 1e-12
    dphi.free()
    env.close()
