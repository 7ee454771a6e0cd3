"""Basis transformation of an operator with an infinite diagonal element: V' = D^T V D is
infinite, with the sign of the product, in the kets of that element's group, and finite
elsewhere; the fragments past a group's last ket add nothing to it."""
import numpy as np
import pytest

from opgen import random_op
from oracle.pyoracle import OracleModelSpace

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


@pytest.mark.parametrize("nrad", [1, 2, 3, 5])
@pytest.mark.parametrize("herm", [1, 0])
def test_transform_infinite_element(ia, nrad, herm):
    print(f"[gpu] transform infinite element nrad={nrad} herm={herm}", flush=True)
    orb = dict(n=[], l=[], j2=[], tz2=[], occ=[], cvq=[])
    for n in range(nrad):
        for l in (0, 1):
            for tz2 in (-1, 1):
                for key, v in zip(orb, (n, l, 1, tz2, 1.0 if n == 0 and l == 0 else 0.0, 0 if n == 0 and l == 0 else 2)):
                    orb[key].append(v)
    ms, orc = ia.ModelSpace(2, orbits=orb), OracleModelSpace(2, orbits=orb)
    ch = next(c for c in ms.channels if c["J"] == 1 and c["tz"] == 0 and c["par"] == 0)  # s s and p p kets
    n, off = ch["n"], ch["off"]
    kets = ms.kets(ms.channels.index(ch))
    blk = [tuple(sorted((ms.orbits[q]["l"], ms.orbits[q]["tz2"]) for q in k)) for k in kets]
    last = max(i for i in range(n) if blk[i] == blk[0])  # the last ket of the first group
    op = random_op(orc, 1, 90 + nrad)
    op["two"][off + last * n + last] = np.inf
    rng = np.random.default_rng(95 + nrad)
    N = len(orb["n"])
    C = np.zeros((N, N))
    for a in range(N):
        for i in range(N):
            if all(orb[q][a] == orb[q][i] for q in ("l", "j2", "tz2")):
                C[i, a] = rng.uniform(0.5, 1.5)  # no D element of the group is 0
    d = ia.Operator(ms, 1, 0.0, op["one"], op["two"]).to_device()
    if herm == 0:
        ia.lib().imsrg_hip_op_set_herm(d.h, 0)
    out = d.TransformToHFBasis(C)
    if herm == 0:
        ia.lib().imsrg_hip_op_set_herm(out.h, 1)  # a host Operator has no such flag
    V = np.asarray(out.to_host().TwoBody)
    block = V[off:off + n * n].reshape(n, n, order="F")
    group = np.array([b == blk[0] for b in blk])
    assert np.all(np.isinf(block[np.ix_(group, group)]))
    rest = np.ones(V.size, bool)
    rest[off:off + n * n] = ~np.outer(group, group).reshape(-1)
    assert np.all(np.isfinite(V[rest]))
    # the sign of D(last, a) D(last, b)
    assert np.array_equal(np.sign(block[np.ix_(group, group)]),
                          np.outer(*2 * [np.sign(block[np.ix_(group, group)][:, 0])]) * np.sign(block[0, 0]))
