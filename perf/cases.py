"""The work that users of imsrg_amd have it do, as cases that can be timed and checked.

Every case goes through the package's public entry points on operators that are resident in HBM (the host-buffer
drop-in: in host memory).  Sizes are those of the repository's benchmark and tests: harmonic-oscillator spaces from
emax = 2 (a scripted check, where launches and latency count) over 4 to 8 (production of small systems, scans) to 10
and 12 (converged calculations), closed-shell and partly filled references, FP64 and mixed precision.

The 64-bit values of ``exact`` come from dense tensors over ordered orbit pairs, in plain torch.
"""
import ctypes
import functools
import math

import numpy as np
import torch

import imsrg_amd as ia

DEV = "cuda" if torch.cuda.is_available() else "cpu"
PRECISION = {"fp64": ia.PREC_FP64, "mixed": ia.PREC_MIXED}
NUCLEI = {"He4": (4, 2), "C12": (12, 6), "N14": (14, 7), "O16": (16, 8), "O18": (18, 8), "Ne20": (20, 10),
          "Si28": (28, 14), "Ca40": (40, 20)}


# ---------------------------------------------------------------------------------------------------------------
# the cases

def listed():
    return [
        # one commutator in the smallest useful space: its time is launches and latency
        {"name": "commutator_e2_fp64", "kind": "commutator", "emax": 2, "ref": "O16", "precision": "fp64"},
        # a small production space with an odd emax
        {"name": "commutator_e5_mixed", "kind": "commutator", "emax": 5, "ref": "O16", "precision": "mixed"},
        # a partly filled reference: fractional occupations give every pp/hh/ph ket a weight
        {"name": "commutator_e7_O18_fp64", "kind": "commutator", "emax": 7, "ref": "O18", "precision": "fp64"},
        # the benchmark's commutator, in both precisions
        {"name": "commutator_e10_fp64", "kind": "commutator", "emax": 10, "ref": "O16", "precision": "fp64"},
        {"name": "commutator_e10_mixed", "kind": "commutator", "emax": 10, "ref": "O16", "precision": "mixed"},
        # a converged space: the largest call
        {"name": "commutator_e12_mixed", "kind": "commutator", "emax": 12, "ref": "O16", "precision": "mixed"},
        # many small independent commutators in one grouped call (a scan over interactions or observables)
        {"name": "batch_e4to7_mixed", "kind": "batch", "pairs": 16, "lo": 4, "hi": 7, "ref": "O16",
         "precision": "mixed"},
        # an observable carried along a flow: the nested commutators of BCH_Transform
        {"name": "bch_transform_e7_fp64", "kind": "bch", "emax": 7, "ref": "O16", "precision": "fp64"},
        # a whole Magnus flow from a Hamiltonian to its decoupled form
        {"name": "magnus_flow_e6_mixed", "kind": "flow", "emax": 6, "ref": "O16", "precision": "mixed"},
        # a Hamiltonian to its Hartree-Fock basis, normal-ordered (the step before every flow)
        {"name": "hartree_fock_e10", "kind": "hf", "emax": 10, "ref": "O16"},
        # normal ordering of an operator over the reference
        {"name": "normal_order_e10", "kind": "normal_order", "emax": 10, "ref": "O16"},
        # the drop-in for a program that keeps its operators in host memory
        {"name": "host_commutator_e8_fp64", "kind": "host", "emax": 8, "ref": "O16", "precision": "fp64"},
    ]


def draw(rng):
    """One more case of the listed ranges; the work grows by about a factor of three with each emax, so a uniform
    emax spreads the sizes over their logarithm."""
    kind = rng.choice(["commutator"] * 5 + ["batch", "bch", "flow", "hf", "normal_order", "transform", "host"])
    top = {"commutator": 12, "bch": 9, "flow": 6, "hf": 10, "normal_order": 11, "transform": 11, "host": 9}
    ref = rng.choice(list(NUCLEI))
    precision = rng.choice(["fp64", "mixed"])
    if kind == "batch":
        lo = rng.randint(3, 7)
        return {"kind": kind, "pairs": rng.randint(2, 20), "lo": lo, "hi": rng.randint(lo, 7), "ref": ref,
                "precision": precision}
    if kind == "flow":
        ref = rng.choice(["He4", "O16", "Ca40"])  # its generator needs a closed shell
    emax = rng.randint(3 if NUCLEI[ref][0] > 16 else 2, top[kind])
    if kind == "commutator" and emax == 12:
        precision = "mixed"  # FP64 at emax = 12 costs more than the largest listed case
    if kind in ("hf", "normal_order", "transform"):
        return {"kind": kind, "emax": emax, "ref": ref}
    return {"kind": kind, "emax": emax, "ref": ref, "precision": precision}


# ---------------------------------------------------------------------------------------------------------------
# the basis: orbits, their occupations and the (J, Tz, parity) channels, in the package's order

class Basis:
    def __init__(self, emax, ref):
        A, Z = NUCLEI[ref]
        orbits = [((N - l) // 2, l, j2, t) for N in range(emax + 1) for l in range(N, -1, -2)
                  for j2 in (2 * l + 1, 2 * l - 1) if j2 > 0 for t in (-1, 1)]
        self.n, self.l, self.j2, self.tz2 = (np.array(v) for v in zip(*orbits))
        self.norb = len(orbits)
        where = {o: i for i, o in enumerate(orbits)}
        self.occ = np.zeros(self.norb)
        left = {-1: float(Z), 1: float(A - Z)}
        for N in range(emax + 1):  # j = l + 1/2 from the largest l down, then j = l - 1/2
            for g in range(2 * N + 1, -2 * N - 1, -4):
                j2, l = abs(g), (abs(g) + (1 if g < 0 else -1)) // 2
                for t in (-1, 1):
                    take = min(left[t], j2 + 1.0)
                    self.occ[where[((N - l) // 2, l, j2, t)]] = take / (j2 + 1.0)
                    left[t] -= take
        self.block = np.array([where[(0, l, j2, t)] for _, l, j2, t in orbits])  # one-body (l, j, tz) block
        p, q = np.triu_indices(self.norb)
        par, tz, same = (self.l[p] + self.l[q]) % 2, (self.tz2[p] + self.tz2[q]) // 2, p == q
        lo, hi = abs(self.j2[p] - self.j2[q]) // 2, (self.j2[p] + self.j2[q]) // 2
        self.nJ = int(self.j2.max()) + 1
        self.channels = []  # (J, kets p, kets q, offset of the n x n block)
        off = 0
        for J in range(self.nJ):
            for t in (-1, 0, 1):
                for pi in (0, 1):
                    k = (lo <= J) & (J <= hi) & (par == pi) & (tz == t) & ~(same & (J % 2 == 1))
                    self.channels.append((J, p[k], q[k], off))
                    off += int(k.sum()) ** 2
        self.size2 = off

    def on(self, a, dtype=None):
        return torch.as_tensor(a, dtype=dtype, device=DEV)


@functools.lru_cache(maxsize=16)
def basis(emax, ref):
    return Basis(emax, ref)


@functools.lru_cache(maxsize=8)
def space(emax, ref):
    """A program keeps one model space for all its operators."""
    return ia.ModelSpace(emax, ref, device=0)


# ---------------------------------------------------------------------------------------------------------------
# operators

def random_operator(B, herm, seed, scale=1.0, one_scale=1.0):
    """(zero, one, two): one- and two-body blocks (R + herm R^T)/sqrt(2 n), R ~ N(0, 1)."""
    g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(n):
        r = torch.randn(n, n, generator=g, device=DEV, dtype=torch.float64)
        return (r + herm * r.T) / math.sqrt(2.0 * max(n, 1))

    one = torch.zeros(B.norb, B.norb, device=DEV, dtype=torch.float64)
    for b in np.unique(B.block):
        k = B.on(np.flatnonzero(B.block == b))
        one[k[:, None], k[None, :]] = one_scale * normal(len(k))
    two = torch.empty(B.size2, device=DEV, dtype=torch.float64)
    for _, p, _, off in B.channels:
        n = len(p)
        two[off:off + n * n] = scale * normal(n).T.reshape(-1)
    return torch.zeros(1, device=DEV, dtype=torch.float64), one, two


def hamiltonian(B, seed):
    """Oscillator energies with off-diagonal one-body elements inside each block, and a random interaction."""
    zero, one, two = random_operator(B, 1, seed, one_scale=0.5)
    one.fill_diagonal_(0.0)
    return zero, one + torch.diag(B.on(10.0 * (2 * B.n + B.l + 1.5))), two


def basis_change(B, seed):
    """An orthogonal change inside each one-body block near 1, as a Hartree-Fock basis is."""
    rng = np.random.default_rng(seed)
    C = np.eye(B.norb)
    for b in np.unique(B.block):
        k = np.flatnonzero(B.block == b)
        q, r = np.linalg.qr(np.eye(len(k)) + 0.2 * rng.normal(size=(len(k), len(k))))
        C[np.ix_(k, k)] = q * np.sign(np.diag(r))
    return C


class _Buffer:
    """`n` doubles of a resident operator from `start`, for torch.  It keeps the operator alive."""

    def __init__(self, op, start, n):
        # an operator's handle begins with its context and its buffer
        buf = ctypes.cast(op.h, ctypes.POINTER(ctypes.c_void_p))[1]
        self.op = op
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f8", "data": (buf + 8 * start, False),
                                         "version": 2}


def resident(op):
    """A resident operator's zero-, one- and two-body parts as the tensors they are in HBM."""
    n1 = op.ms.norb ** 2
    parts = ((0, 1), (8, n1), (8 + (n1 + 7) // 8 * 8, op.ms.tbsize))
    return tuple(torch.as_tensor(_Buffer(op, a, n), device=DEV) for a, n in parts)


def _flat(values):
    zero, one, two = values
    return zero, one.T.reshape(-1), two  # one-body matrices are column-major


def to_device(ms, herm, values):
    op = ia.DeviceOperator(ms, herm)
    for to, v in zip(resident(op), _flat(values)):
        to.copy_(v)
    return op


# ---------------------------------------------------------------------------------------------------------------
# inputs of a case, from its seed

OMEGA = 0.02  # size of the BCH case's Omega: about 18 nested commutators, as in an early step of a flow


def _inputs(case, seed):
    """The operators of a case as (emax, herm, values)."""
    kind = case["kind"]
    seed = 1000 * int(seed)
    if kind == "batch":
        out = []
        for i in range(case["pairs"]):
            e = case["lo"] + i % (case["hi"] - case["lo"] + 1)
            B = basis(e, case["ref"])
            out += [(e, -1, random_operator(B, -1, seed + 2 * i)), (e, 1, random_operator(B, 1, seed + 2 * i + 1))]
        return out
    e, B = case["emax"], basis(case["emax"], case["ref"])
    if kind in ("commutator", "host"):
        return [(e, -1, random_operator(B, -1, seed)), (e, 1, random_operator(B, 1, seed + 1))]
    if kind == "bch":
        return [(e, 1, hamiltonian(B, seed)), (e, -1, random_operator(B, -1, seed + 1, OMEGA, OMEGA))]
    return [(e, 1, hamiltonian(B, seed))]


def prepare(case, seed):
    kind = case["kind"]
    state = {"kind": kind, "precision": PRECISION[case.get("precision", "fp64")]}
    given = _inputs(case, seed)
    if kind == "host":
        ms = space(case["emax"], case["ref"])
        state["ops"] = [ia.Operator(ms, h, float(z[0]), one.cpu().numpy(), two.cpu().numpy())
                        for _, h, (z, one, two) in given]
        return state
    ops = [to_device(space(e, case["ref"]), h, v) for e, h, v in given]
    torch.cuda.synchronize()
    if kind in ("commutator", "batch"):
        pairs = [(x, y, ia.DeviceOperator(x.ms, 1)) for x, y in zip(ops[::2], ops[1::2])]
        state["pairs"] = pairs
        state["out"] = tuple(t for _, _, z in pairs for t in resident(z))
    else:
        state["ops"] = ops
        state["to"] = ia.DeviceOperator(ops[0].ms, 1)
        state["out"] = resident(state["to"])
    if kind == "transform":
        state["C"] = np.asfortranarray(basis_change(basis(case["emax"], case["ref"]), seed))
    return state


def run(state):
    kind, precision = state["kind"], state["precision"]
    if kind == "commutator":
        x, y, z = state["pairs"][0]
        ia.Commutator.CommutatorScalarScalar(x, y, precision=precision, out=z)
        return state["out"]
    if kind == "batch":
        ia.Commutator.CommutatorScalarScalarBatched(state["pairs"], precision=precision)
        return state["out"]
    if kind == "host":
        z = ia.Commutator.CommutatorScalarScalar(*state["ops"], precision=precision)
        return z.ZeroBody, z.OneBody, z.TwoBody
    if kind == "bch":
        ia.BCH.BCH_Transform(*state["ops"], out=state["to"], precision=precision)
        return state["out"]
    if kind == "flow":
        h, e0, eta, ncomm = ia.IMSRGSolver.Solve_magnus_euler(state["ops"][0], ds=0.5, smax=20.0, eta_criterion=1e-6,
                                                              mode=1, transform_thr=1e-8, precision=precision)
        return {"H": resident(h), "E0": e0, "eta": eta, "commutators": ncomm}
    if kind == "hf":
        hf = ia.HartreeFock(state["ops"][0]).Solve()
        hf.GetNormalOrderedH(out=state["to"])
        return {"H": state["out"], "C": hf.C, "F": hf.F, "energies": hf.energies, "EHF": [hf.EHF, hf.e1hf, hf.e2hf]}
    if kind == "normal_order":
        state["ops"][0].DoNormalOrdering(out=state["to"])
    else:
        state["ops"][0].TransformToHFBasis(state["C"], out=state["to"])
    return state["out"]


# ---------------------------------------------------------------------------------------------------------------
# what a pass cannot do without

@functools.lru_cache(maxsize=64)
def _commutator_flops(emax, ref):
    """The pp/hh products of every channel (X W Y over kets without an unequal pair of occupations, both triangles
    from one product) and the particle-hole products of every cross-coupled channel."""
    B = basis(emax, ref)
    occ = B.occ
    w = [np.abs((1 - occ[p]) * (1 - occ[q]) - occ[p] * occ[q]) > 1e-12 for _, p, q, _ in B.channels]
    pphh = sum(2.0 * len(k) ** 2 * int(k.sum()) for k in w)
    p, q = np.triu_indices(B.norb)
    lo, hi = abs(B.j2[p] - B.j2[q]) // 2, (B.j2[p] + B.j2[q]) // 2
    group = 2 * (abs(B.tz2[p] - B.tz2[q]) // 2) + (B.l[p] + B.l[q]) % 2
    ph = abs(occ[p] - occ[q]) > 1e-12
    total = 0.0
    for J in range(B.nJ):
        for g in range(4):
            k = (lo <= J) & (J <= hi) & (group == g)
            total += 8.0 * int(k.sum()) ** 2 * int((k & ph).sum())
    return pphh + total


def _size(emax, ref):
    B = basis(emax, ref)
    return 8.0 * (B.size2 + B.norb ** 2)


def work(case):
    kind, ref = case["kind"], case["ref"]
    if kind == "batch":
        es = [case["lo"] + i % (case["hi"] - case["lo"] + 1) for i in range(case["pairs"])]
        return {"bytes": sum(3 * _size(e, ref) for e in es), "flops": sum(_commutator_flops(e, ref) for e in es)}
    e = case["emax"]
    size = _size(e, ref)
    if kind in ("commutator", "host"):
        return {"bytes": 3 * size, "flops": _commutator_flops(e, ref)}
    if kind == "bch":  # about 18 nested commutators
        return {"bytes": 3 * size, "flops": 18 * _commutator_flops(e, ref)}
    if kind == "flow":  # about 250 nested commutators
        return {"bytes": 2 * size, "flops": 250 * _commutator_flops(e, ref)}
    B = basis(e, ref)
    if kind == "normal_order":
        return {"bytes": 2 * size, "flops": 2.0 * B.norb ** 2}
    flops = 0.0  # D^T V D with D block diagonal over pairs of one-body blocks
    for _, p, q, _ in B.channels:
        key = np.minimum(B.block[p], B.block[q]) * B.norb + np.maximum(B.block[p], B.block[q])
        flops += 4.0 * len(p) * float((np.unique(key, return_counts=True)[1] ** 2).sum())
    return {"bytes": 2 * size, "flops": flops}


# ---------------------------------------------------------------------------------------------------------------
# 64-bit values: the same quantities from dense tensors over ordered orbit pairs.  T^J[p, q, r, s] are the
# antisymmetrised elements <pq|T|rs>_J with sqrt(2) for each pair of equal orbits.

@functools.lru_cache(maxsize=4)
def sixj(nj, nJ):
    """{ja jb J; jc jd K} for half-integer j = (2 i + 1)/2, i < nj, and J, K < nJ, as [ia, ib, J, ic, id, K]."""
    i, k = np.arange(nj) * 2 + 1, np.arange(nJ) * 2
    a, b, c, d, e, f = np.meshgrid(i, i, k, i, i, k, indexing="ij")
    ok = np.ones(a.shape, bool)
    for x, y, z in ((a, b, c), (a, e, f), (d, b, f), (d, e, c)):
        ok &= (abs(x - y) <= z) & (z <= x + y)
    a, b, c, d, e, f = (v[ok] for v in (a, b, c, d, e, f))
    fact = np.cumprod(np.concatenate([[1], np.arange(1, 4 * 2 * nj + 8)]).astype(np.longdouble))
    pre = np.ones(len(a), np.longdouble)
    for x, y, z in ((a, b, c), (a, e, f), (d, b, f), (d, e, c)):
        pre *= fact[(x + y - z) // 2] * fact[(x - y + z) // 2] * fact[(y + z - x) // 2] / fact[(x + y + z) // 2 + 1]
    low = [(a + b + c) // 2, (a + e + f) // 2, (d + b + f) // 2, (d + e + c) // 2]
    high = [(a + b + d + e) // 2, (b + c + e + f) // 2, (a + c + d + f) // 2]
    tmin, tmax = np.max(low, axis=0), np.min(high, axis=0)
    total = np.zeros(len(a), np.longdouble)
    for s in range(int((tmax - tmin).max()) + 1 if len(a) else 0):
        t = tmin + s
        m = np.flatnonzero(t <= tmax)
        t = t[m]
        den = np.ones(len(m), np.longdouble)
        for v in low:
            den *= fact[t - v[m]]
        for v in high:
            den *= fact[v[m] - t]
        total[m] += np.where(t % 2 == 0, 1, -1) * fact[t + 1] / den
    out = np.zeros(ok.shape)
    out[ok] = (np.sqrt(pre) * total).astype(np.float64)
    return out


def dense(B, two, J):
    """T^J as a matrix over ordered pairs."""
    n = B.norb
    T = torch.zeros(n * n, n * n, device=DEV, dtype=torch.float64)
    for K, p, q, off in B.channels:
        if K != J or not len(p):
            continue
        m = two[off:off + len(p) ** 2].view(len(p), len(p)).T
        s = B.on(np.where(p == q, math.sqrt(2.0), 1.0))
        m = m * s[:, None] * s[None, :]
        x = B.on(1.0 - 2.0 * (((B.j2[p] + B.j2[q]) // 2 + 1 + J) % 2))
        pq, qp = B.on(p * n + q), B.on(q * n + p)
        T[pq[:, None], pq[None, :]] = m
        T[qp[:, None], pq[None, :]] = x[:, None] * m
        T[pq[:, None], qp[None, :]] = m * x[None, :]
        T[qp[:, None], qp[None, :]] = x[:, None] * m * x[None, :]
    return T


def pack(B, two, J, T):
    """T^J into the package's layout."""
    for K, p, q, off in B.channels:
        if K != J or not len(p):
            continue
        pq = B.on(p * B.norb + q)
        s = B.on(np.where(p == q, math.sqrt(2.0), 1.0))
        m = T[pq[:, None], pq[None, :]] / s[:, None] / s[None, :]
        two[off:off + len(p) ** 2] = m.T.reshape(-1)


def _sign(x):
    return 1.0 - 2.0 * (x % 2)


def commutator64(B, X, Y, hx, hy):
    """(zero, one, two) of [X, Y] in the IMSRG(2) truncation."""
    n, nJ = B.norb, B.nJ
    hz = -1 if hx == hy else 1
    X1, Y1 = X[1], Y[1]
    occ, jf = B.on(B.occ), B.on(B.j2 + 1.0)
    same = B.on(B.block[:, None] == B.block[None, :])
    tx, ty = [dense(B, X[2], J) for J in range(nJ)], [dense(B, Y[2], J) for J in range(nJ)]
    four = (n, n, n, n)
    zero = (jf * occ * torch.diagonal(X1 @ Y1 - Y1 @ X1)).sum()
    one = X1 @ Y1 - Y1 @ X1
    # particles and holes of the ordered pairs
    pp, hh = torch.outer(1 - occ, 1 - occ).reshape(-1), torch.outer(occ, occ).reshape(-1)
    nab = torch.outer(occ, 1 - occ) * same
    tz = []
    for J in range(nJ):
        x, y = tx[J], ty[J]
        mpp, mhh = 0.5 * (x * pp) @ y, 0.5 * (x * hh) @ y
        if hx != hy:
            zero = zero + 0.5 * (2 * J + 1) * (hh[:, None] * x * pp * y.T).sum()
        mpp, mhh = mpp + hz * mpp.T, mhh + hz * mhh.T
        z = mpp - mhh
        for m, w in ((mpp, occ), (mhh, 1 - occ)):  # sum over c of M(c i, c j)
            one = one + (2 * J + 1) * torch.einsum("c,cicj->ij", w, m.view(four)) / jf[:, None] * same
        for u, t, s in ((X1, y, 1.0), (Y1, x, -1.0)):
            a = u @ t.view(n, n ** 3)  # u on the first orbit, then on each of the others
            z = z + s * a.view(n * n, n * n)
            a = torch.matmul(u, t.view(n, n, n * n))
            z = z + s * a.view(n * n, n * n)
            a = torch.matmul(u.T, t.view(n * n, n, n))
            z = z - s * a.view(n * n, n * n)
            z = z - s * (t.view(n ** 3, n) @ u).view(n * n, n * n)
            # one-body: n_a (1 - n_b) [u_ab T_{bi aj} - u_ba T_{ai bj}]
            t4 = t.view(four)
            v = torch.einsum("ab,biaj->ij", nab * u, t4) - torch.einsum("ab,aibj->ij", nab * u.T, t4)
            one = one + s * (2 * J + 1) * v / jf[:, None] * same
        tz.append(z)
    # particle-hole term: cross-coupled elements, their product, and back
    jj = B.on((B.j2 - 1) // 2)
    s6 = B.on(sixj(int(B.j2.max() + 1) // 2, nJ))
    ia_, ib_, ic_, id_ = jj[:, None, None, None], jj[None, :, None, None], jj[None, None, :, None], jj[None, None, None, :]
    j2, w = B.on(B.j2), (occ[:, None] - occ[None, :]).reshape(-1)
    for K in range(nJ):
        xb, yb = torch.zeros(four, device=DEV, dtype=torch.float64), torch.zeros(four, device=DEV, dtype=torch.float64)
        for J in range(nJ):
            s = s6[:, :, K, :, :, J]
            if not bool((s != 0).any()):
                continue
            s = (2 * J + 1) * s[ic_, id_, ia_, ib_]  # {ja jb K; jc jd J} over [c, d, a, b]
            xb -= s * tx[J].view(four).permute(0, 3, 2, 1)
            yb -= hy * s * ty[J].view(four).permute(0, 3, 2, 1)
        zb = (xb.view(n * n, n * n) * w) @ yb.view(n * n, n * n).T
        zb = (zb + hz * zb.T).view(four)
        del xb, yb
        for J in range(nJ):
            s = s6[:, :, J, :, :, K]
            if not bool((s != 0).any()):
                continue
            s = s[ia_, ib_, ic_, id_] * (2 * K + 1)  # over [i, j, k, l]
            z = tz[J].view(four)
            z += s * zb.permute(0, 3, 2, 1)
            s = s6[:, :, J, :, :, K][ib_, ia_, ic_, id_] * (2 * K + 1)
            z -= _sign((j2[:, None] + j2[None, :]) // 2 - J)[:, :, None, None] * s * zb.permute(3, 0, 2, 1)
    two = torch.zeros_like(X[2])
    for J in range(nJ):
        pack(B, two, J, tz[J])
    return zero.reshape(1), one, two


def norm64(B, T):
    one = (T[1] ** 2 * B.on(B.j2 + 1.0)[:, None]).sum()
    two = sum((2 * J + 1) ** 2 * (T[2][off:off + len(p) ** 2] ** 2).sum() for J, p, _, off in B.channels)
    return math.sqrt(float(one + two))


def bch64(B, H, W, thr=1e-9, most=40):
    """exp(W) H exp(-W) with the truncation of BCH_Transform's default rule."""
    out, nested = [t.clone() for t in H], H
    ny = norm64(B, W)
    eps = norm64(B, H) * math.exp(-2 * ny) * thr / (2 * ny)
    fact = 1.0
    for i in range(1, most + 1):
        nested = commutator64(B, W, nested, -1, 1)
        fact /= i
        eps *= i + 1
        for o, t in zip(out, nested):
            o += fact * t
        if norm64(B, nested) < eps:
            break
    return tuple(out)


def normal_order64(B, H):
    occ, jf = B.on(B.occ), B.on(B.j2 + 1.0)
    zero, one = H[0] + (jf * occ * torch.diagonal(H[1])).sum(), H[1].clone()
    same = B.on(B.block[:, None] == B.block[None, :])
    for J in range(B.nJ):
        t = dense(B, H[2], J).view((B.norb,) * 4)
        v = (2 * J + 1) * torch.diagonal(t, dim1=1, dim2=3) @ occ  # sum over h of T_{ah bh} n_h
        zero = zero + 0.5 * (torch.diagonal(v) * occ).sum()
        one = one + v / jf[:, None] * same
    return zero, one, H[2].clone()


def transform64(B, H, C):
    C = B.on(C)
    n = B.norb
    two = torch.zeros_like(H[2])
    for J in range(B.nJ):
        t = dense(B, H[2], J)
        t = (C.T @ t.view(n, n ** 3)).view(n, n, n * n)
        t = torch.matmul(C.T, t).view(n * n, n, n)
        t = torch.matmul(C.T, t).view(n ** 3, n)
        pack(B, two, J, (t @ C).view(n * n, n * n))
    return H[0].clone(), C.T @ H[1] @ C, two


def hartree_fock64(B, H):
    """The self-consistent basis by the package's iteration: the density mixed with a fifth of the last one."""
    n, occ, jf = B.norb, B.occ, B.j2 + 1.0
    mono = torch.zeros((n,) * 4, device=DEV, dtype=torch.float64)
    for J in range(B.nJ):
        mono += (2 * J + 1) * dense(B, H[2], J).view((n,) * 4)
    same = B.on(B.block[:, None] == B.block[None, :])
    h1 = H[1].cpu().numpy()

    def field(rho):
        v = torch.einsum("iajb,ab->ij", mono, B.on(rho) * same) * same
        v = torch.triu(v / B.on(jf)[:, None])
        return (v + torch.triu(v, 1).T).cpu().numpy()

    def density(C):
        return (C * occ) @ C.T

    C, e = np.eye(n), np.diag(h1).copy()
    rho = density(C)
    v = field(rho)
    for _ in range(100):
        last, C, e = e, np.zeros((n, n)), np.zeros(n)
        for b in np.unique(B.block):
            k = np.flatnonzero(B.block == b)
            e[k], C[np.ix_(k, k)] = np.linalg.eigh((h1 + v)[np.ix_(k, k)])
        C *= np.where(np.diag(C) < 0, -1.0, 1.0)
        rho = 0.8 * density(C) + 0.2 * rho
        v = field(rho)
        if np.linalg.norm(e - last) / n < 1e-8:
            break
    else:
        return None
    del mono
    e1, e2 = float((rho * jf[:, None] * h1).sum()), float(0.5 * (rho * jf[:, None] * v).sum())
    F = h1 + v
    two = transform64(B, H, C)[2]
    return {"H": (np.array([e1 + e2]), (C.T @ F @ C).T.reshape(-1), two), "C": C, "F": F, "energies": e,
            "EHF": [e1 + e2, e1, e2]}


def exact(case, seed):
    kind = case["kind"]
    if kind == "flow":
        return None  # hundreds of commutators
    top = {"commutator": 8, "host": 8, "bch": 7, "batch": 7}.get(kind, 10)
    if max(case.get("emax", 0), case.get("hi", 0)) > top:
        return None  # over 20 seconds or over the card's memory
    given = [(basis(e, case["ref"]), h, v) for e, h, v in _inputs(case, seed)]
    B, _, H = given[0]
    if kind in ("commutator", "batch"):
        return tuple(t for (b, hx, x), (_, hy, y) in zip(given[::2], given[1::2])
                     for t in _flat(commutator64(b, x, y, hx, hy)))
    if kind == "host":
        zero, one, two = commutator64(B, H, given[1][2], -1, 1)
        return float(zero), one, two
    if kind == "bch":
        return _flat(bch64(B, H, given[1][2]))
    if kind == "normal_order":
        return _flat(normal_order64(B, H))
    if kind == "transform":
        return _flat(transform64(B, H, basis_change(B, seed)))
    return hartree_fock64(B, H)
