"""Performance cases: what programs on tennetlib_amd spend their time in.

Two-site DMRG and TDVP on MPS are a loop over bonds of an environment update,
a Krylov solve made of products of the projected operator, and a truncating
factorisation; TTN optimisation is the same over tree nodes.  The cases are
those parts one by one, through the C ABI and the Python entry points that
programs call, over bond dimensions from the first sweeps of a ramp (16) to
the largest the framework is run at (4096), and whole calls of each kind:

  product    one product of the two-site projected operator (tn_env_matvec)
  move       the environment moved one bond right and back (position_), with
             the product at each position, as a sweep steps through a chain
  eig        the Lanczos solve of one DMRG update (contract_phi, krylov_eig)
  expm       the Krylov exponential of one TDVP update (contract_phi,
             krylov_expm), complex tensors
  truncate   the truncating factorisation of one update (replacebond)
  qn         product and factorisation of one update of a Hubbard chain whose
             tensors are block-sparse in (N_up, N_dn)
  dmrg       dmrg_ from a random product state over a bond-dimension ramp
  tdvp       tdvpsweep_ steps from a random product state
  ttn        optimize_ of a random-field chain on the default binary tree

Models are the framework's own: Heisenberg and XXZ chains (MPO bond 5), the
J1-J2 cylinder of width 6 (MPO bond 17 to 20), the Hubbard chain (MPO bond 6,
d = 4) and the random-field Heisenberg chain on a tree.
"""

import ctypes
import functools
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path("tennetlib.jl_amd").resolve()))

import tennetlib_amd as T  # noqa: E402

PRECISION = {"fp64": 0, "fp32": 1, "bf16x3": 2}
# GEMM rates (flop/s) that bound what a drawn case may cost
RATE = {"fp64": 50e12, "fp32": 130e12, "bf16x3": 300e12, "complex": 30e12}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # first sweeps of a ramp on a chain: a few launches per product
        dict(name="product chi16", kind="product", model="chain", prec="fp64", chil=16, chir=16),
        # BF16x3 form of the wide-MPO cylinder at a middle bond dimension
        dict(name="product bf16x3 chi2048 w20", kind="product", model="cylinder", prec="bf16x3", chil=2048, chir=2048),
        # the mixed-precision form of the headline workload, chi = 4096
        dict(name="product fp32 chi4096 w20", kind="product", model="cylinder", prec="fp32", chil=4096, chir=4096),
        # one step of a cylinder sweep in FP64, odd bond dimensions
        dict(name="move chi255 w20", kind="move", model="cylinder", chil=255, chir=253),
        # Lanczos of one update where the N = 100 Heisenberg chain saturates
        dict(name="eig chi185", kind="eig", model="chain", prec="fp64", chil=185, chir=181, kdim=5, maxiter=2),
        # Krylov exponential of one TDVP update after some entanglement growth
        dict(name="expm complex chi200", kind="expm", model="chain", chil=200, chir=200, dt=0.05),
        # factorisation of the same Heisenberg bond: a 370-row density matrix
        dict(name="truncate chi185", kind="truncate", complex=False, d=2, chil=185, chir=181, maxdim=185, left=True),
        # factorisation of a large bulk bond: a 4096-row density matrix
        dict(name="truncate chi2048", kind="truncate", complex=False, d=2, chil=2048, chir=2048, maxdim=2048,
             left=False),
        # one bond of a QN-conserving Hubbard chain, tens of sectors per link
        dict(name="qn hubbard chi500", kind="qn", prec="fp64", sites=16, chi=500, left=True),
        # a short DMRG ramp from scratch, the smallest whole calculation
        dict(name="dmrg heisenberg n20", kind="dmrg", sites=20, prec="fp64", chi=64),
        # real-time evolution of a spin chain, complex tensors
        dict(name="tdvp xxz n16", kind="tdvp", sites=16, chi=48, steps=3, dt=0.05),
        # one random-field instance of a many-instance TTN batch
        dict(name="ttn random field n32", kind="ttn", sites=32, chi=24, sweeps=1),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, uniform in the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = 0.9 * _product_flops(4096, 4096, 2, 20, 20) / RATE["fp32"]
    kind = rng.choice(["product", "product", "move", "eig", "expm", "truncate", "truncate", "qn", "dmrg", "tdvp",
                       "ttn"])
    while True:
        if kind == "product":
            prec = rng.choice(["fp64", "fp32", "bf16x3", "complex"])
            model = "chain" if prec == "complex" else rng.choice(["chain", "cylinder", "hubbard"])
            chil = _log(rng, 12, 512 if prec == "complex" else 4096 if model != "hubbard" else 1200)
            c = dict(kind=kind, model=model, prec=prec, chil=chil,
                     chir=max(8, int(chil * rng.choice([1, 1, rng.uniform(0.5, 1)]))))
            d, w = {"chain": (2, 5), "cylinder": (2, 20), "hubbard": (4, 6)}[model]
            cost = _product_flops(chil, c["chir"], d, w, w) * (4 if prec == "complex" else 1) / RATE[prec]
        elif kind == "move":
            chil = _log(rng, 16, 900)
            c = dict(kind=kind, model=rng.choice(["chain", "cylinder"]), chil=chil,
                     chir=max(12, int(chil * rng.uniform(0.6, 1))))
            cost = 0.0
        elif kind == "eig":
            chil = _log(rng, 16, 700)
            c = dict(kind=kind, model="chain", prec=rng.choice(["fp64", "fp64", "fp32"]), chil=chil,
                     chir=max(12, int(chil * rng.uniform(0.6, 1))), kdim=rng.choice([3, 5]), maxiter=rng.choice([1, 2]))
            cost = 0.0
        elif kind == "expm":
            chil = _log(rng, 12, 400)
            c = dict(kind=kind, model="chain", chil=chil, chir=max(8, int(chil * rng.uniform(0.6, 1))),
                     dt=rng.choice([0.02, 0.05, 0.1]))
            cost = 0.0
        elif kind == "truncate":
            cx = rng.random() < 0.3
            d = rng.choice([2, 2, 4])
            chil = _log(rng, 16, (512 if cx else 4096) // d)
            chir = min((512 if cx else 4096) // d, max(12, int(chil * rng.uniform(0.7, 1.3))))
            c = dict(kind=kind, complex=cx, d=d, chil=chil, chir=chir,
                     maxdim=max(8, int(chil * rng.uniform(0.5, 1))), left=rng.random() < 0.5)
            cost = 0.0
        elif kind == "qn":
            c = dict(kind=kind, prec=rng.choice(["fp64", "fp32", "bf16x3"]), sites=rng.choice([12, 14, 16]),
                     chi=_log(rng, 60, 500), left=rng.random() < 0.5)
            cost = 0.0
        elif kind == "dmrg":
            c = dict(kind=kind, sites=rng.randint(12, 24), prec=rng.choice(["fp64", "fp32"]), chi=_log(rng, 24, 80))
            cost = 0.0
        elif kind == "tdvp":
            c = dict(kind=kind, sites=rng.randint(10, 16), chi=_log(rng, 16, 48), steps=rng.randint(1, 3),
                     dt=rng.choice([0.02, 0.05, 0.1]))
            cost = 0.0
        else:
            c = dict(kind=kind, sites=rng.randint(12, 32), chi=_log(rng, 8, 24), sweeps=1)
            cost = 0.0
        if cost <= most:
            return c


# ---------------------------------------------------------------------------
# models and states
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _cylinder():
    return T.j1j2_cylinder_mpo(6, 12, 1.0, 0.5)


def _mpo(model, n):
    """MPO of n sites: a whole chain, or n bulk sites of the cylinder with its
    outer channels closed by fixed vectors."""
    if model == "chain":
        return T.xxz_mpo(n, 1.0, 1.0)
    if model == "hubbard":
        return T.hubbard_mpo(n)
    first = 36 - n // 2
    Ws = list(_cylinder()[first:first + n])
    rng = np.random.default_rng(11)
    Ws[0] = np.tensordot(rng.uniform(-1, 1, Ws[0].shape[0]), Ws[0], axes=([0], [0]))[None]
    Ws[-1] = np.tensordot(Ws[-1], rng.uniform(-1, 1, Ws[-1].shape[3]), axes=([3], [0]))[..., None]
    return [np.ascontiguousarray(W) for W in Ws]


def _random(rng, shape, cx):
    a = rng.standard_normal(shape)
    return a + 1j * rng.standard_normal(shape) if cx else a


def _edges(c, seed):
    """Four sites whose middle two sit between bonds chil and chir; the outer
    two are random edges, so the environments of position 2 are dense."""
    rng = np.random.default_rng(seed)
    cx = c["prec"] == "complex"
    Ws = _mpo(c["model"], 4)
    d, chil, chir = Ws[0].shape[1], c["chil"], c["chir"]
    A = [_random(rng, (1, d, chil), cx) / math.sqrt(d), _random(rng, (chil, d, 1), cx),
         _random(rng, (1, d, chir), cx), _random(rng, (chir, d, 1), cx) / math.sqrt(d)]
    return A, Ws, 2


def _window(c, seed, cx=False):
    """A mixed-canonical random MPS around its centre bond b, whose outer links
    have dimensions chil and chir and fall off toward the ends as fast as the
    physical dimension allows."""
    rng = np.random.default_rng(seed)
    d, chil, chir = 2, c["chil"], c["chir"]
    nl = max(1, math.ceil(math.log(chil, d) - 1e-9))
    nr = max(2, math.ceil(math.log(chir, d) - 1e-9))
    left = [min(d ** k, chil) for k in range(nl + 1)]
    right = [min(d ** k, chir) for k in range(nr + 1)]
    left[-1], right[-1] = chil, chir
    A = []
    for k in range(nl):
        q, _ = np.linalg.qr(_random(rng, (left[k] * d, left[k + 1]), cx))
        A.append(q.reshape(left[k], d, left[k + 1]))
    mid = min(chil, chir) * d if min(chil, chir) < 4 else max(chil, chir)
    mid = min(mid, d * chil, d * chir)
    A.append(_random(rng, (chil, d, mid), cx) / math.sqrt(chil * d * mid))
    q, _ = np.linalg.qr(_random(rng, (d * chir, mid), cx))
    A.append(np.ascontiguousarray(q.T).reshape(mid, d, chir))
    for k in range(nr, 0, -1):
        q, _ = np.linalg.qr(_random(rng, (d * right[k - 1], right[k]), cx))
        A.append(np.ascontiguousarray(q.T).reshape(right[k], d, right[k - 1]))
    A[nl] /= np.linalg.norm(A[nl])
    return [np.ascontiguousarray(a) for a in A], _mpo(c["model"], len(A)), nl + 1


def _vector(shape, seed, cx):
    g = torch.Generator(device="cuda").manual_seed(seed)
    v = torch.randn(shape, generator=g, device="cuda", dtype=torch.complex128 if cx else torch.float64)
    return v / torch.linalg.vector_norm(v)


def _orthonormal(n, r, rng):
    """n x r dense matrix with orthonormal columns: cosine transforms between
    random signs, r of its columns in random order."""
    i = torch.arange(n, device="cuda")
    x = ((2 * i[:, None] + 1) * i[None, :]) % (4 * n)
    F = math.sqrt(2.0 / n) * torch.cos(x.double() * (math.pi / (2 * n)))
    F[:, 0] /= math.sqrt(2.0)
    s1, s2 = (torch.from_numpy(rng.choice([-1.0, 1.0], n)).cuda() for _ in range(2))
    cols = torch.from_numpy(rng.permutation(n)[:r]).cuda()
    return s1[:, None] * (F @ (s2[:, None] * F.T[:, cols]))


def _spectrum(c):
    """Singular values of a two-site tensor that maxdim cuts: they fall
    stretched-exponentially, in multiplets of three as spin multiplets do, with
    the cut between two multiplets."""
    m, n = c["chil"] * c["d"], c["chir"] * c["d"]
    r, k = min(m, n), min(c["maxdim"], m, n)
    i = np.arange(r)
    s = 10.0 ** (-5.0 * (np.floor((i - k) / 3.0) * 3.0 / k + 1.0 + 3.0 / k) ** 0.7)
    s /= np.linalg.norm(s)
    return s, k


def _two_site_tensor(c, seed):
    """phi = U diag(s) V^H (m x n, unit norm) and its factors."""
    rng = np.random.default_rng(seed)
    m, n = c["chil"] * c["d"], c["chir"] * c["d"]
    s, k = _spectrum(c)
    r = len(s)
    U, V = _orthonormal(m, r, rng), _orthonormal(n, r, rng)
    if c["complex"]:
        U, V = U.to(torch.complex128), V.to(torch.complex128)
        for F, rows in ((U, m), (V, n)):
            F *= torch.polar(torch.ones(rows, dtype=torch.float64, device="cuda"),
                             torch.from_numpy(rng.uniform(0, 2 * math.pi, rows)).cuda())[:, None]
    st = torch.from_numpy(s).cuda()
    return (U * st) @ V.mH, U, st, V, k


# Hubbard chain links: sector dimensions around the most likely fillings ------
@functools.lru_cache(maxsize=None)
def _sectors(sites, chi):
    """For links 0..sites of a half-filled Hubbard chain, {(N_up, N_dn): dim}
    in ascending order; the centre bond b = sites / 2 is left free."""
    half, b = sites // 2, sites // 2
    qs = T.hubbard_qns()

    def target(k):
        frac = k * half / sites
        g = {(u, v): math.exp(-((u - frac) ** 2 + (v - frac) ** 2) / 1.6)
             for u in range(min(k, half) + 1) for v in range(min(k, half) + 1)}
        tot = sum(g.values())
        return {q: max(1, round(chi * x / tot)) for q, x in g.items() if chi * x / tot >= 0.5}

    links = [None] * (sites + 1)
    links[0], links[sites] = {(0, 0): 1}, {(half, half): 1}
    for k in range(1, b):
        t, prev = target(k), links[k - 1]
        room = {q: sum(prev.get((q[0] - s[0], q[1] - s[1]), 0) for s in qs) for q in t}
        links[k] = {q: min(t[q], room[q]) for q in sorted(t) if room[q]}
    for k in range(sites - 1, b, -1):
        t, nxt = target(k), links[k + 1]
        room = {q: sum(nxt.get((q[0] + s[0], q[1] + s[1]), 0) for s in qs) for q in t}
        links[k] = {q: min(t[q], room[q]) for q in sorted(t) if room[q]}
    t = target(b)
    reach = {q: min(sum(links[b - 1].get((q[0] - s[0], q[1] - s[1]), 0) for s in qs),
                    sum(links[b + 1].get((q[0] + s[0], q[1] + s[1]), 0) for s in qs)) for q in t}
    links[b] = {q: min(t[q], reach[q]) for q in sorted(t) if reach[q]}
    return links


def _offsets(link):
    out, o = {}, 0
    for q, n in link.items():
        out[q] = (o, n)
        o += n
    return out


def _hubbard_state(c, seed):
    """Block-sparse mixed-canonical MPS around b and a block-sparse two-site
    tensor with falling singular values in every sector."""
    rng = np.random.default_rng(seed)
    sites, b = c["sites"], c["sites"] // 2
    links = _sectors(sites, c["chi"])
    qs = T.hubbard_qns()
    off = [_offsets(x) for x in links]
    dim = [sum(x.values()) for x in links]
    A = []
    for k in range(1, sites + 1):
        a = np.zeros((dim[k - 1], 4, dim[k]))
        if k <= b:
            for q, (o, n) in off[k].items():
                rows = [(o2, n2, s) for s in range(4)
                        for o2, n2 in [off[k - 1].get((q[0] - qs[s][0], q[1] - qs[s][1]), (0, 0))] if n2]
                f, _ = np.linalg.qr(rng.standard_normal((sum(x[1] for x in rows), n)))
                i = 0
                for o2, n2, s in rows:
                    a[o2:o2 + n2, s, o:o + n] = f[i:i + n2]
                    i += n2
        else:
            for q, (o, n) in off[k - 1].items():
                cols = [(o2, n2, s) for s in range(4)
                        for o2, n2 in [off[k].get((q[0] + qs[s][0], q[1] + qs[s][1]), (0, 0))] if n2]
                f, _ = np.linalg.qr(rng.standard_normal((sum(x[1] for x in cols), n)))
                i = 0
                for o2, n2, s in cols:
                    a[o:o + n, s, o2:o2 + n2] = f[i:i + n2].T
                    i += n2
        A.append(a)
    phi = np.zeros((dim[b - 1], 4, 4, dim[b + 1]))
    flat = phi.reshape(dim[b - 1] * 4, 4 * dim[b + 1])
    for rows, cols in _blocks(c):
        r = min(len(rows), len(cols))
        s = rng.uniform(0.7, 1.3) * 10.0 ** (-6.0 * (np.arange(r) / max(r, 2)) ** 0.7)
        u = rng.standard_normal((len(rows), r)) / math.sqrt(len(rows))
        v = rng.standard_normal((r, len(cols))) / math.sqrt(len(cols))
        flat[np.ix_(rows, cols)] = (u * s) @ v * math.sqrt(r)
    phi /= np.linalg.norm(phi)
    labels = [[q for q, n in x.items() for _ in range(n)] for x in links]
    return A, T.hubbard_mpo(sites), b, phi, labels


def _blocks(c):
    """Row and column indices (of phi as a matrix) of every sector of bond b."""
    b = c["sites"] // 2
    links = _sectors(c["sites"], c["chi"])
    qs = T.hubbard_qns()
    ql = [q for q, n in links[b - 1].items() for _ in range(n)]
    qr = [q for q, n in links[b + 1].items() for _ in range(n)]
    rows, cols = {}, {}
    for a, q in enumerate(ql):
        for s in range(4):
            rows.setdefault((q[0] + qs[s][0], q[1] + qs[s][1]), []).append(4 * a + s)
    for t in range(4):
        for i, q in enumerate(qr):
            cols.setdefault((q[0] - qs[t][0], q[1] - qs[t][1]), []).append(t * len(qr) + i)
    return [(rows[q], cols[q]) for q in sorted(rows) if q in cols]


# ---------------------------------------------------------------------------
# states and passes
# ---------------------------------------------------------------------------
def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _environment(A, Ws, b, dtype=None):
    env = T.StateEnvs(A, Ws, dtype=dtype)
    T.set_nsite_(env, 2)
    T.position_(env, b)
    env.set_orthocenter(b)
    return env


def prepare(case, seed):
    c, kind = case, case["kind"]
    st = {"case": c}
    if kind == "product":
        A, Ws, b = _edges(c, seed)
        st["env"] = _environment(A, Ws, b)
        d = Ws[0].shape[1]
        st["v"] = _vector((c["chil"], d, d, c["chir"]), seed, c["prec"] == "complex")
        st["out"] = torch.empty_like(st["v"])
    elif kind == "move":
        A, Ws, b = _window(c, seed)
        st["env"], st["b"] = _environment(A, Ws, b), b
        st["v"] = [_vector((A[k - 1].shape[0], 2, 2, A[k].shape[2]), seed + k, False) for k in (b, b + 1)]
        st["out"] = [torch.empty_like(v) for v in st["v"]]
    elif kind in ("eig", "expm"):
        cx = kind == "expm"
        A, Ws, b = _window(c, seed, cx)
        st["env"], st["b"] = _environment(A, Ws, b), b
        st["phi"] = torch.empty((c["chil"], 2, 2, c["chir"]), device="cuda",
                                dtype=torch.complex128 if cx else torch.float64)
    elif kind == "truncate":
        d, dt = c["d"], np.complex128 if c["complex"] else np.float64
        st["phi"] = _two_site_tensor(c, seed)[0].reshape(c["chil"], d, d, c["chir"]).contiguous()
        # only the outer links of the two sites matter: replacebond writes both
        A = [np.ones((1, d, c["chil"]), dt), np.ones((c["chil"], d, 1), dt), np.ones((1, d, c["chir"]), dt),
             np.ones((c["chir"], d, 1), dt)]
        st["env"], st["b"] = T.StateEnvs(A, _mpo("chain" if d == 2 else "hubbard", 4)), 2
        st["out"], st["weights"] = torch.empty_like(st["phi"]), (ctypes.c_double * c["maxdim"])()
    elif kind == "qn":
        A, Ws, b, phi, labels = _hubbard_state(c, seed)
        env = _environment(A, Ws, b)
        site = np.array([q for _ in range(c["sites"]) for q in T.hubbard_qns()], np.int32).reshape(-1)
        link = np.array([q for x in labels for q in x], np.int32).reshape(-1)
        pi = ctypes.POINTER(ctypes.c_int)
        env.ctx.check(env.ctx.lib.tn_env_set_qn(env.h, 2, site.ctypes.data_as(pi), link.ctypes.data_as(pi)))
        env.nq = 2
        st["env"], st["b"], st["phi"] = env, b, torch.from_numpy(phi).cuda()
        st["product"], st["out"] = torch.empty_like(st["phi"]), torch.empty_like(st["phi"])
        st["weights"] = (ctypes.c_double * c["chi"])()
    elif kind in ("dmrg", "tdvp"):
        rng = np.random.default_rng(seed)
        vs = [_random(rng, 2, kind == "tdvp") for _ in range(c["sites"])]
        st["psi"] = T.product_state([v / np.linalg.norm(v) for v in vs],
                                    np.complex128 if kind == "tdvp" else np.float64)
        st["mpo"] = T.xxz_mpo(c["sites"], 1.0, 0.5 if kind == "tdvp" else 1.0)
    else:
        from tennetlib_amd.batch import random_field_chain
        rng = np.random.default_rng(seed)
        st["model"] = random_field_chain(c["sites"], rng.uniform(-1, 1, c["sites"]))
        st["psi"] = T.default_randomTTN(c["sites"], c["chi"], seed=seed)
        st["path"] = T.default_sweeppath(st["psi"])
    torch.cuda.synchronize()
    return st


def _padded(weights, n):
    out = np.zeros(n)
    w = np.sort(np.asarray(weights, dtype=np.float64))[::-1][:n]
    out[:len(w)] = w
    return out


def _truncate(env, b, phi, out, c, maxdim, weights):
    """The factorisation of an update; returns the truncated two-site tensor and
    the kept weights, which do not depend on the gauge of the two factors."""
    err, kept = ctypes.c_double(), ctypes.c_long()
    env.ctx.check(env.ctx.lib.tn_replacebond(env.h, b, _ptr(phi), int(c["left"]), maxdim, 1, 1e-14, 0.0, 1,
                                             ctypes.byref(err), weights, maxdim, ctypes.byref(kept)))
    env.ctx.check(env.ctx.lib.tn_env_contract_phi(env.h, b, _ptr(out)))
    return out, _padded(weights[:min(kept.value, maxdim)], maxdim)


def run(state):
    c, kind = state["case"], state["case"]["kind"]
    if kind == "product":
        env, prec = state["env"], PRECISION["fp64" if c["prec"] == "complex" else c["prec"]]
        env.ctx.check(env.ctx.lib.tn_env_matvec(env.h, _ptr(state["v"]), _ptr(state["out"]), prec))
        return state["out"]
    if kind == "move":
        env, b = state["env"], state["b"]
        for pos, i in ((b + 1, 1), (b, 0)):
            T.position_(env, pos)
            env.ctx.check(env.ctx.lib.tn_env_matvec(env.h, _ptr(state["v"][i]), _ptr(state["out"][i]), 0))
        return state["out"]
    if kind == "eig":
        env, e = state["env"], ctypes.c_double()
        env.ctx.check(env.ctx.lib.tn_env_contract_phi(env.h, state["b"], _ptr(state["phi"])))
        env.ctx.check(env.ctx.lib.tn_krylov_eig(env.h, _ptr(state["phi"]), c["kdim"], c["maxiter"], 1e-14,
                                                PRECISION[c["prec"]], ctypes.byref(e), None))
        return e.value, state["phi"]
    if kind == "expm":
        env = state["env"]
        env.ctx.check(env.ctx.lib.tn_env_contract_phi(env.h, state["b"], _ptr(state["phi"])))
        env.ctx.check(env.ctx.lib.tn_krylov_expm(env.h, _ptr(state["phi"]), 0.0, -0.5 * c["dt"], 30, 100, 1e-12, 0,
                                                 None))
        return state["phi"]
    if kind == "truncate":
        return _truncate(state["env"], state["b"], state["phi"], state["out"], c, c["maxdim"], state["weights"])
    if kind == "qn":
        env = state["env"]
        env.ctx.check(env.ctx.lib.tn_env_matvec(env.h, _ptr(state["phi"]), _ptr(state["product"]),
                                                PRECISION[c["prec"]]))
        return state["product"], *_truncate(env, state["b"], state["phi"], state["out"], c, c["chi"],
                                            state["weights"])
    if kind == "dmrg":
        env = T.StateEnvs(state["psi"], state["mpo"])
        ramp = [16, max(16, c["chi"] // 2), c["chi"]]
        sw = T.dmrg_(env, T.make_dmrg_params(maxdim=ramp, nsweeps=[1, 1, 1], cutoff=1e-10), 2, solver_krylovdim=3,
                     solver_maxiter=2, precision=c["prec"], outputlevel=0)
        env.close()
        return np.array(sw.energy), np.stack([_padded(w, c["chi"]) for w in sw.lasteigs])
    if kind == "tdvp":
        eng = T.TDVPEngine(state["psi"], state["mpo"])
        for _ in range(c["steps"]):
            T.tdvpsweep_(eng, -1j * c["dt"], 2, maxdim=c["chi"], cutoff=1e-12, outputlevel=0)
        eng.sysenv.close()
        return np.array(eng.swdata.energy), np.stack([_padded(w, c["chi"]) for w in eng.swdata.lasteigs])
    env = T.StateEnvsTTN(state["psi"], state["model"])
    sw = T.optimize_(env, T.make_optimize_params(maxdim=[c["chi"]], nsweeps=[c["sweeps"]], cutoff=1e-14),
                     state["path"], outputlevel=0)
    psi = env.psi
    env.close()
    # the state up to the gauge of its links: the entanglement weights of the three links of its centre
    A = psi.tensors[psi.orthocenter]
    return np.array(sw.energy), [np.linalg.svd(np.moveaxis(A, k, 0).reshape(A.shape[k], -1), compute_uv=False) ** 2
                                 for k in range(3)]


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------
def _product_flops(chil, chir, d, wl, wr):
    """The two GEMMs and the MPO contraction between them."""
    return 2.0 * chil * chir * d * d * (wl * chil + wr * chir) + 4.0 * chil * chir * d ** 3 * wl * wr


def _product_bytes(chil, chir, d, wl, wr, size):
    return size * (wl * chil * chil + wr * chir * chir) + 16.0 * d * d * chil * chir * max(1, size // 8)


def _svd_flops(m, n, k):
    """Density matrix, tridiagonalisation, kept eigenvectors, other factor."""
    p, q = min(m, n), max(m, n)
    return 2.0 * p * p * q / 2 + 4.0 / 3.0 * p ** 3 + 2.0 * p * p * k + 2.0 * m * n * k


def _bond_dims(sites, chi, d=2):
    return [min(d ** min(k, sites - k), chi) for k in range(sites + 1)]


def work(case):
    c, kind = case, case["kind"]
    if kind == "product":
        d, w = {"chain": (2, 5), "cylinder": (2, 20), "hubbard": (4, 6)}[c["model"]]
        size = {"fp64": 8, "complex": 16}.get(c["prec"], 4)
        return {"bytes": _product_bytes(c["chil"], c["chir"], d, w, w, size),
                "flops": _product_flops(c["chil"], c["chir"], d, w, w) * (4 if c["prec"] == "complex" else 1)}
    if kind in ("move", "eig", "expm"):
        d, w = 2, 20 if c["model"] == "cylinder" else 5
        a, b = c["chil"], c["chir"]
        nops, cx = {"move": 2, "eig": c.get("kdim", 0) + (2 if c.get("maxiter") == 2 else 0), "expm": 8}[kind], kind == "expm"
        f = nops * _product_flops(a, b, d, w, w)
        y = _product_bytes(a, b, d, w, w, 8) + 8.0 * (a * a + b * b) * d
        if kind == "move":
            m = max(a, b)
            f += 2.0 * w * d * (a * a * m + a * m * m) + 2.0 * w * d * (b * b * m + b * m * m)
            y += 8.0 * w * 2 * m * m
        return {"bytes": y * (2 if cx else 1), "flops": f * (4 if cx else 1)}
    if kind == "truncate":
        m, n, cx = c["chil"] * c["d"], c["chir"] * c["d"], c["complex"]
        k = min(c["maxdim"], m, n)
        return {"bytes": 8.0 * (2 * m * n + k * (m + n)) * (2 if cx else 1), "flops": _svd_flops(m, n, k) * (4 if cx else 1)}
    if kind == "qn":
        sec = _blocks(c)
        links, b = _sectors(c["sites"], c["chi"]), c["sites"] // 2
        qs = T.hubbard_qns()
        f = 0.0
        for q, n in links[b - 1].items():
            for s in qs:
                for t in qs:
                    r = links[b + 1].get((q[0] + s[0] + t[0], q[1] + s[1] + t[1]), 0)
                    f += 2.0 * 6 * n * r * (n + r)
        f += sum(_svd_flops(len(x), len(y), min(len(x), len(y)) / 2) for x, y in sec)
        env = sum(n * n for k in (b - 1, b + 1) for n in links[k].values())
        return {"bytes": 8.0 * (6 * env + 4 * sum(len(x) * len(y) for x, y in sec)), "flops": f}
    if kind in ("dmrg", "tdvp"):
        tot, byt = 0.0, 0.0
        for chi in ([16, max(16, c["chi"] // 2), c["chi"]] if kind == "dmrg" else [c["chi"] // 2] * c["steps"]):
            dims = _bond_dims(c["sites"], chi)
            for b in range(1, c["sites"]):
                l, r = dims[b - 1], dims[b + 1]
                tot += 2 * ((5 if kind == "dmrg" else 8) * _product_flops(l, r, 2, 5, 5) + _svd_flops(2 * l, 2 * r, min(l, r)))
                byt += 2 * _product_bytes(l, r, 2, 5, 5, 8)
        return {"bytes": byt * (2 if kind == "tdvp" else 1), "flops": tot * (4 if kind == "tdvp" else 1)}
    n, chi = c["sites"], c["chi"]
    inner = max(1, n - 2)
    return {"bytes": 2.0 * c["sweeps"] * inner * 8 * 3 * 6 * chi * chi,
            "flops": 2.0 * c["sweeps"] * inner * 7 * 3 * 2.0 * 6 * chi ** 4 / 4}


# ---------------------------------------------------------------------------
# tolerances and 64-bit references
# ---------------------------------------------------------------------------
def tolerance(case):
    """About four times what the same pass with its sums in another order, or
    the 64-bit reference, differs by over these ranges."""
    kind, prec = case["kind"], case.get("prec", "fp64")
    if kind in ("product", "eig", "qn") and prec == "bf16x3":
        return {"rel": 4e-5}   # 16-bit split mantissas: 9e-6 at chi = 2048
    if kind in ("product", "eig", "qn") and prec == "fp32":
        return {"rel": 3e-5}   # sums over w chi = 81920 terms: 7e-6 at chi = 4096
    if kind == "dmrg":
        return {"rel": 1e-5}   # early ramp sweeps move with rounding; maxdim cuts multiplets
    if kind in ("tdvp", "ttn"):
        return {"rel": 1e-6}
    if kind in ("truncate", "qn"):
        return {"rel": 2e-9}   # weights below the cut mix at rounding over gap: 2e-10 at 4096 rows
    return {"rel": 4e-13 if kind in ("eig", "expm") else 4e-14}


def _local(A, Ws, b):
    """The two-site projected operator of an MPS at bond b, in 64 bits."""
    dt = torch.complex128 if any(np.iscomplexobj(a) for a in A) else torch.float64
    A = [torch.from_numpy(np.ascontiguousarray(a)).cuda().to(dt) for a in A]
    W = [torch.from_numpy(np.ascontiguousarray(w)).cuda().to(dt) for w in Ws]
    one = torch.ones((1, 1, 1), dtype=dt, device="cuda")
    L, R = one, one
    for k in range(b - 1):  # L[w, a', a]
        X = torch.tensordot(L, A[k], dims=([2], [0]))                 # w a' s b
        X = torch.tensordot(X, W[k], dims=([0, 2], [0, 2]))           # a' b s' w'
        L = torch.tensordot(A[k].conj(), X, dims=([0, 1], [0, 2])).permute(2, 0, 1).contiguous()
    for k in range(len(A) - 1, b, -1):  # R[w, b, b']
        X = torch.tensordot(A[k], R, dims=([2], [1]))                 # a s w b'
        X = torch.tensordot(X, W[k], dims=([1, 2], [2, 3]))           # a b' w s'
        R = torch.tensordot(X, A[k].conj(), dims=([1, 3], [2, 1])).permute(1, 0, 2).contiguous()
    op = torch.tensordot(W[b - 1], W[b], dims=([3], [0]))             # w s' s t' t w2

    def apply(v):
        chil, d, e, chir = v.shape
        X = torch.tensordot(L, v, dims=([2], [0]))                    # w a' s t b
        X = torch.tensordot(op, X, dims=([0, 2, 4], [0, 2, 3]))       # s' t' w2 a' b
        X = torch.tensordot(X, R, dims=([2, 4], [0, 1]))              # s' t' a' b'
        return X.permute(2, 0, 1, 3).contiguous()

    return apply


def _centre(A, b):
    x = torch.tensordot(torch.from_numpy(A[b - 1]).cuda(), torch.from_numpy(A[b]).cuda(), dims=([2], [0]))
    return x.contiguous()


def _dot(x, y):
    return torch.sum(x.conj() * y)


def _lanczos(apply, v, kdim, maxiter):
    """Lowest Ritz pair after maxiter cycles of kdim vectors, three fifths of the
    Ritz vectors kept at a restart with the residual direction, every vector
    orthogonalised against all others."""
    V = [v / torch.linalg.vector_norm(v)]
    HV, cycle = [], 1

    def extend():
        HV.append(apply(V[-1]))
        w = HV[-1].clone()
        for _ in range(2):
            for x in V:
                w -= _dot(x, w) * x
        return w

    while True:
        while True:
            w = extend()
            if len(V) == kdim:
                break
            V.append(w / torch.linalg.vector_norm(w))
        Hm = torch.stack([torch.stack([_dot(x, y) for y in HV]) for x in V]).cpu()
        th, U = torch.linalg.eigh(0.5 * (Hm + Hm.mH))

        def mix(S, j):
            return sum(U[i, j].item() * S[i] for i in range(len(S)))

        if cycle == maxiter:
            x = mix(V, 0)
            return th[0].item(), x / torch.linalg.vector_norm(x)
        keep = max(1, min(3 * kdim // 5, kdim - 1))
        V, HV = [mix(V, j) for j in range(keep)] + [w / torch.linalg.vector_norm(w)], [mix(HV, j) for j in range(keep)]
        cycle += 1


def _exponential(apply, v, t):
    """exp(t H) v from Taylor series over short sub-steps."""
    n = 8
    for _ in range(n):
        term, v = v, v.clone()
        for k in range(1, 40):
            term = apply(term) * (t / (n * k))
            v += term
            if torch.linalg.vector_norm(term).item() < 1e-18 * torch.linalg.vector_norm(v).item():
                break
    return v


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "product":
        A, Ws, b = _edges(c, seed)
        v = _vector((c["chil"], Ws[0].shape[1], Ws[0].shape[1], c["chir"]), seed, c["prec"] == "complex")
        return _local(A, Ws, b)(v)
    if kind == "move":
        A, Ws, b = _window(c, seed)
        return [_local(A, Ws, k)(_vector((A[k - 1].shape[0], 2, 2, A[k].shape[2]), seed + k, False))
                for k in (b, b + 1)]
    if kind == "eig":
        A, Ws, b = _window(c, seed)
        e, _ = _lanczos(_local(A, Ws, b), _centre(A, b), c["kdim"], c["maxiter"])
        return e, None  # the Ritz vector's sign is a convention
    if kind == "expm":
        A, Ws, b = _window(c, seed, True)
        return _exponential(_local(A, Ws, b), _centre(A, b), -0.5j * c["dt"])
    if kind == "truncate":
        _, U, s, V, k = _two_site_tensor(c, seed)
        nrm = torch.linalg.vector_norm(s[:k])
        out = (U[:, :k] * (s[:k] / nrm)) @ V[:, :k].mH
        return out.reshape(c["chil"], c["d"], c["d"], c["chir"]), _padded((s[:k] ** 2).cpu().numpy(), c["maxdim"])
    if kind == "qn":
        A, Ws, b, phi, _ = _hubbard_state(c, seed)
        M = phi.reshape(phi.shape[0] * 4, -1)
        parts = [np.linalg.svd(M[np.ix_(r, q)], full_matrices=False) for r, q in _blocks(c)]
        cut = np.sort(np.concatenate([p[1] for p in parts]))[::-1][:c["chi"] + 1]
        low = cut[c["chi"]] if len(cut) > c["chi"] else 0.0
        out, kept = np.zeros_like(M), []
        for (r, q), (u, s, v) in zip(_blocks(c), parts):
            n = int(np.sum(s > low))
            out[np.ix_(r, q)] = (u[:, :n] * s[:n]) @ v[:n]
            kept.append(s[:n])
        kept = np.concatenate(kept)
        return (_local(A, Ws, b)(torch.from_numpy(phi).cuda()), (out / np.linalg.norm(kept)).reshape(phi.shape),
                _padded(kept ** 2, c["chi"]))
    return None
