"""bf16x3 pp/hh GEMM against the oracle at numbers of k stages around its ring of three and
at the edges of its tiles, in each order of the tiles."""
import numpy as np
import pytest

from opgen import random_op
from oracle.pyoracle import TERMS, OracleModelSpace

pytestmark = pytest.mark.gpu
TOL = 2e-6  # operands to 2^-26, 32 products summed in FP32: 33 roundings of 2^-24


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


@pytest.mark.parametrize("nrad", [1, 3, 4, 5, 6, 7, 8, 10, 12])
def test_pphh_b3_stages(ia, nrad):
    print(f"[gpu] bf16x3 pp/hh stages nrad={nrad}", flush=True)
    orb = dict(n=[], l=[], j2=[], tz2=[], occ=[], cvq=[])
    for n in range(nrad):
        for l, j2 in ((0, 1), (1, 1), (1, 3)):
            for tz2 in (-1, 1):
                h = l == 0 and n == 0
                for key, v in zip(orb, (n, l, j2, tz2, 1.0 if h else 0.0, 0 if h else 2)):
                    orb[key].append(v)
    ms, orc = ia.ModelSpace(3, orbits=orb), OracleModelSpace(3, orbits=orb)
    for hx, hy in ((-1, 1), (-1, -1)):
        X, Y = random_op(orc, hx, 90 + nrad), random_op(orc, hy, 60 + nrad)
        dX = ia.Operator(ms, hx, 0.0, X["one"], X["two"]).to_device()
        dY = ia.Operator(ms, hy, 0.0, Y["one"], Y["two"]).to_device()
        R = orc.commutator(X, Y, TERMS["comm222_pp_hhss"])["two"]
        for order in (0, 1, 2):
            ms.set_tuning(pphh_small_tile_max=0, pphh_order=order)
            Z = ia.Commutator.CommutatorScalarScalar(dX, dY, TERMS["comm222_pp_hhss"], precision=ia.PREC_MIXED).to_host()
            assert np.max(np.abs(Z.TwoBody - R)) <= TOL * max(np.max(np.abs(R)), 1e-300)
