"""comm222_ph against the oracle where the inverse Pandya kernel's items change shape:
bras whose elements of Zbar exceed one work-group's LDS (ranges of k; with any of its
sizes), groups of many kets of one class, both work-group sizes, and a space without holes (Zbar = 0)."""
import numpy as np
import pytest

from opgen import random_op
from oracle.pyoracle import TERMS, OracleModelSpace

pytestmark = pytest.mark.gpu
TOL = 1e-12       # the FP64 bar of the parity tests, relative max-abs
TOL_FP32 = 2e-6   # operands rounded to FP32 and 32 products summed in it: 33 roundings of 2^-24


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


@pytest.mark.parametrize("nrad,lj,holes", [
    (2, [(0, 1), (1, 1), (1, 3)], [(0, 0, 1)]),
    (1, [(0, 1), (1, 3), (3, 7), (4, 7)], [(0, 1, 3), (0, 4, 7)]),
    (3, [(0, 1), (1, 1), (1, 3)], []),
    (6, [(0, 1), (1, 1), (1, 3), (2, 3), (2, 5)], [(0, 0, 1), (0, 2, 5)]),
    (8, [(0, 1), (1, 1), (1, 3), (2, 3), (2, 5)], [(0, 0, 1), (0, 2, 5)]),
    (12, [(0, 1), (1, 1), (1, 3), (2, 3), (2, 5)], [(0, 0, 1), (0, 2, 5)]),
])
def test_ph_items(ia, nrad, lj, holes):
    print(f"[gpu] inverse Pandya items nrad={nrad} lj={lj} holes={holes}", flush=True)
    orb = dict(n=[], l=[], j2=[], tz2=[], occ=[], cvq=[])
    for n in range(nrad):
        for l, j2 in lj:
            for tz2 in (-1, 1):
                h = (n, l, j2) in holes
                for key, v in zip(orb, (n, l, j2, tz2, 1.0 if h else 0.0, 0 if h else 2)):
                    orb[key].append(v)
    emax = max(j2 for _, j2 in lj)
    ms, orc = ia.ModelSpace(emax, orbits=orb), OracleModelSpace(emax, orbits=orb)
    for hx, hy in ((-1, 1), (1, 1)):
        X, Y = random_op(orc, hx, 5), random_op(orc, hy, 6)
        dX = ia.Operator(ms, hx, 0.0, X["one"], X["two"]).to_device()
        dY = ia.Operator(ms, hy, 0.0, Y["one"], Y["two"]).to_device()
        R = orc.commutator(X, Y, TERMS["comm222_phss"])["two"]
        for prec, tol in ((0, TOL), (1, TOL_FP32)):
            Z = ia.Commutator.CommutatorScalarScalar(dX, dY, TERMS["comm222_phss"], precision=prec).to_host()
            assert np.max(np.abs(Z.TwoBody - R)) <= tol * max(np.max(np.abs(R)), 1e-300)
