"""ph GEMM against the oracle at the edges of its tiles and k stages: channels of one ket
up to a few past 128, and numbers of ph kets that leave remainders of a 32-k stage."""
import numpy as np
import pytest

from opgen import random_op
from oracle.pyoracle import TERMS, OracleModelSpace

pytestmark = pytest.mark.gpu
TOL = 1e-12      # the FP64 bar of the parity tests, relative max-abs
TOL_FP32 = 2e-6  # operands rounded to FP32 and 32 products summed in it: 33 roundings of 2^-24


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


@pytest.mark.parametrize("nrad,nholes", [(1, 1), (2, 1), (3, 2), (5, 1), (7, 3), (8, 2), (11, 4)])
def test_ph_sizes(ia, nrad, nholes):
    print(f"[gpu] ph GEMM sizes nrad={nrad} nholes={nholes}", flush=True)
    orb = dict(n=[], l=[], j2=[], tz2=[], occ=[], cvq=[])
    for n in range(nrad):
        for l, j2 in ((0, 1), (1, 1), (1, 3)):
            for tz2 in (-1, 1):
                h = l == 0 and n < nholes
                for key, v in zip(orb, (n, l, j2, tz2, 1.0 if h else 0.0, 0 if h else 2)):
                    orb[key].append(v)
    ms, orc = ia.ModelSpace(3, orbits=orb), OracleModelSpace(3, orbits=orb)
    for hx, hy in ((-1, 1), (-1, -1)):
        X, Y = random_op(orc, hx, 3 + nrad), random_op(orc, hy, 40 + nrad)
        dX = ia.Operator(ms, hx, 0.0, X["one"], X["two"]).to_device()
        dY = ia.Operator(ms, hy, 0.0, Y["one"], Y["two"]).to_device()
        R = orc.commutator(X, Y, TERMS["comm222_phss"])["two"]
        for prec, tol in ((0, TOL), (1, TOL_FP32)):
            Z = ia.Commutator.CommutatorScalarScalar(dX, dY, TERMS["comm222_phss"], precision=prec).to_host()
            assert np.max(np.abs(Z.TwoBody - R)) <= tol * max(np.max(np.abs(R)), 1e-300)
