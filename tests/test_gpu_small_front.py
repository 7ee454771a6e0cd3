"""Commutators around the sizes where the first launch stops taking comm122 and the small
pp/hh tiles, with and without a second stream, against the oracle."""
import numpy as np
import pytest

from opgen import random_op
from oracle.pyoracle import ALL_TERMS, TERMS, OracleModelSpace

pytestmark = pytest.mark.gpu
TOL = 1e-12  # the FP64 bar of the parity tests, relative max-abs


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


@pytest.mark.parametrize("emax,A,Z", [(1, 4, 2), (2, 4, 2), (3, 16, 8), (5, 16, 8), (6, 16, 8), (6, 40, 20)])
def test_small_front(ia, emax, A, Z):
    print(f"[gpu] small front emax={emax} A={A} Z={Z}", flush=True)
    ms, orc = ia.ModelSpace(emax, (A, Z)), OracleModelSpace(emax, A, Z)
    X, Y = random_op(orc, -1, 7), random_op(orc, 1, 8)
    dX = ia.Operator(ms, -1, X["zero"], X["one"], X["two"]).to_device()
    dY = ia.Operator(ms, 1, Y["zero"], Y["one"], Y["two"]).to_device()
    for terms in (ALL_TERMS, TERMS["comm122ss"], TERMS["comm222_pp_hhss"] | TERMS["comm122ss"]):
        R = orc.commutator(X, Y, terms)
        for overlap in (0, 1, 2):
            ms.set_tuning(overlap_pphh=overlap)
            Z_ = ia.Commutator.CommutatorScalarScalar(dX, dY, terms).to_host()
            for x, y in ((np.asarray(Z_.OneBody), R["one"]), (np.asarray(Z_.TwoBody), R["two"])):
                assert np.max(np.abs(x - y)) <= TOL * max(np.max(np.abs(y)), 1e-300)
