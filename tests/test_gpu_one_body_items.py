"""One-body terms against the oracle where the comm221 work items are cut: numbers of
(c, J) entries that are not multiples of 4, of particle orbits that are not multiples of
16, occupations between 0 and 1 (an orbit in both lists), and no holes at all."""
import numpy as np
import pytest

from opgen import random_op
from oracle.pyoracle import ALL_TERMS, OracleModelSpace

pytestmark = pytest.mark.gpu
TOL = 1e-12  # the FP64 bar of the parity tests, relative max-abs


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


@pytest.mark.parametrize("nrad,lj,holes", [
    (1, [(0, 1)], {(0, 0, 1): 1.0}),
    (2, [(0, 1), (1, 1), (1, 3)], {(0, 0, 1): 1.0, (0, 1, 3): 0.5}),
    (4, [(0, 1), (3, 7)], {(0, 0, 1): 1.0, (0, 3, 7): 1.0, (1, 3, 7): 0.25}),
    (3, [(0, 1), (1, 1), (1, 3), (2, 5)], {}),
    (4, [(0, 1), (1, 3), (2, 3), (5, 11)], {(0, 0, 1): 1.0, (0, 1, 3): 1.0, (0, 5, 11): 1.0}),
])
def test_one_body_items(ia, nrad, lj, holes):
    print(f"[gpu] one-body items nrad={nrad} lj={lj} holes={holes}", flush=True)
    orb = dict(n=[], l=[], j2=[], tz2=[], occ=[], cvq=[])
    for n in range(nrad):
        for l, j2 in lj:
            for tz2 in (-1, 1):
                occ = holes.get((n, l, j2), 0.0)
                for key, v in zip(orb, (n, l, j2, tz2, occ, 0 if occ else 2)):
                    orb[key].append(v)
    emax = max(j2 for _, j2 in lj)
    ms, orc = ia.ModelSpace(emax, orbits=orb), OracleModelSpace(emax, orbits=orb)
    for hx, hy in ((-1, 1), (1, 1)):
        X, Y = random_op(orc, hx, 9), random_op(orc, hy, 10)
        dX = ia.Operator(ms, hx, X["zero"], X["one"], X["two"]).to_device()
        dY = ia.Operator(ms, hy, Y["zero"], Y["one"], Y["two"]).to_device()
        R = orc.commutator(X, Y, ALL_TERMS)
        Z = ia.Commutator.CommutatorScalarScalar(dX, dY, ALL_TERMS).to_host()
        one = np.asarray(R["one"]).reshape(Z.OneBody.shape)
        scale = max(np.max(np.abs(R["two"])), np.max(np.abs(one)))
        assert np.max(np.abs(Z.OneBody - one)) <= TOL * scale
        assert np.max(np.abs(Z.TwoBody - R["two"])) <= TOL * scale
