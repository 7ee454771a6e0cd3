"""The ph term against the oracle on a basis whose inverse Pandya tables alone take more than
the smaller LDS sizes of a work-group, so that its items are cut to fit the largest."""
import numpy as np
import pytest

from oracle import pyoracle
from oracle.pyoracle import TERMS, OracleModelSpace

pytestmark = pytest.mark.gpu
TOL = 1e-12  # the FP64 bar of the parity tests, relative max-abs


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


def test_ph_term_on_a_large_basis(ia):
    print("[gpu] ph term emax=12 A=132", flush=True)
    ms = ia.ModelSpace(12, (132, 50))
    X = ia.DeviceOperator(ms, -1).fill_random(-1, 91)
    Y = ia.DeviceOperator(ms, 1).fill_random(1, 92)
    Z = ia.Commutator.CommutatorScalarScalar(X, Y, TERMS["comm222_phss"]).to_host()
    print("[gpu] done, now the oracle", flush=True)
    ops = [dict(zero=o.ZeroBody, one=np.asfortranarray(o.OneBody), two=np.asarray(o.TwoBody), herm=o.herm)
           for o in (X.to_host(), Y.to_host())]
    pyoracle.use_blas(True)
    try:
        R = OracleModelSpace(12, 132, 50).commutator(*ops, TERMS["comm222_phss"])["two"]
    finally:
        pyoracle.use_blas(False)
    scale = max(R.max(), -R.min())
    R -= Z.TwoBody
    assert max(R.max(), -R.min()) <= TOL * scale
