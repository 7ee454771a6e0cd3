"""The ph term with an Inf or NaN in the first element of an operand, which the Pandya
gather reads in place of terms that do not exist: it reaches the elements that are sums
over it, as in the oracle, and no others."""
import numpy as np
import pytest

from opgen import random_op
from oracle.pyoracle import TERMS, OracleModelSpace

pytestmark = pytest.mark.gpu
TOL = 1e-12  # the FP64 bar of the parity tests, relative max-abs


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


@pytest.mark.parametrize("emax", [2, 4, 7])
@pytest.mark.parametrize("which", ["X", "Y"])
def test_pandya_not_finite(ia, emax, which):
    print(f"[gpu] ph term, first element of {which} not finite, emax={emax}", flush=True)
    ms, orc = ia.ModelSpace(emax, "O16"), OracleModelSpace(emax, 16, 8)
    ops = {"X": random_op(orc, 1, 71), "Y": random_op(orc, 1, 72)}
    ops[which]["two"][0] = np.nan
    dX = ia.Operator(ms, 1, 0.0, ops["X"]["one"], ops["X"]["two"]).to_device()
    dY = ia.Operator(ms, 1, 0.0, ops["Y"]["one"], ops["Y"]["two"]).to_device()
    Z = np.asarray(ia.Commutator.CommutatorScalarScalar(dX, dY, TERMS["comm222_phss"]).to_host().TwoBody)
    R = orc.commutator(ops["X"], ops["Y"], TERMS["comm222_phss"])["two"]
    good = np.isfinite(R)
    assert 0 < np.count_nonzero(~good) < 0.5 * R.size
    assert np.array_equal(np.isfinite(Z), good)
    assert np.max(np.abs(Z[good] - R[good])) <= TOL * np.max(np.abs(R[good]))
