"""Block-sparse basis transformation against the oracle at group sizes around its 16-column
and 4-ket fragments, past its largest group (dense path), and without Hermiticity."""
import numpy as np
import pytest

from opgen import random_op
from oracle.pyoracle import OracleModelSpace

pytestmark = pytest.mark.gpu
TOL = 1e-13  # as for the other sizes: sums of at most 81 products in another order


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


@pytest.mark.parametrize("nrad", [1, 2, 4, 5, 8, 9])
@pytest.mark.parametrize("herm", [1, -1, 0])
def test_transform_group_sizes(ia, nrad, herm):
    print(f"[gpu] transform groups nrad={nrad} herm={herm}", flush=True)
    orb = dict(n=[], l=[], j2=[], tz2=[], occ=[], cvq=[])
    for n in range(nrad):
        for l, j2 in ((0, 1), (1, 1), (1, 3)):
            for tz2 in (-1, 1):
                for key, v in zip(orb, (n, l, j2, tz2, 1.0 if n == 0 and l == 0 else 0.0, 0 if n == 0 and l == 0 else 2)):
                    orb[key].append(v)
    ms, orc = ia.ModelSpace(3, orbits=orb), OracleModelSpace(3, orbits=orb)
    op = random_op(orc, herm if herm else 1, 70 + nrad)
    rng = np.random.default_rng(80 + nrad)
    if herm == 0:  # nothing symmetric about it
        op["one"] = op["one"] * rng.uniform(0.5, 1.5, op["one"].shape)
        op["two"] = op["two"] * rng.uniform(0.5, 1.5, op["two"].shape)
    N = len(orb["n"])
    C = np.zeros((N, N))
    for a in range(N):
        for i in range(N):
            if all(orb[q][a] == orb[q][i] for q in ("l", "j2", "tz2")):
                C[i, a] = rng.standard_normal() / np.sqrt(nrad)
    d = ia.Operator(ms, op["herm"], 0.0, op["one"], op["two"]).to_device()
    if herm == 0:
        ia.lib().imsrg_hip_op_set_herm(d.h, 0)
    out = d.TransformToHFBasis(C)
    if herm == 0:
        ia.lib().imsrg_hip_op_set_herm(out.h, 1)  # a host Operator has no such flag
    got, ref = out.to_host(), orc.transform_basis(op, C)
    for x, y in ((np.asarray(got.OneBody), ref["one"]), (np.asarray(got.TwoBody), ref["two"])):
        assert np.max(np.abs(x - y)) <= TOL * max(np.max(np.abs(y)), 1e-300)
