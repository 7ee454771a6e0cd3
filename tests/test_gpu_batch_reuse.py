"""One list of contexts in batches of changing precision and terms: the batch keeps its
workspaces and tables, and a call finds the contents that another precision (FP32 or FP64
Zbar, Xbar and Ybar in the same memory) and other terms have left there."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


def test_batch_keeps_nothing_of_the_last_call(ia):
    print("[gpu] batch reuse", flush=True)
    from imsrg_amd import ALL_TERMS, PREC_FP64, PREC_MIXED, PREC_SPLIT, TERMS
    spaces = [ia.ModelSpace(4, "O16"), ia.ModelSpace(3, "He4"), ia.ModelSpace(4, "Ca40")]
    pairs = [(ia.DeviceOperator(m, -1).fill_random(-1, 10 + i), ia.DeviceOperator(m, 1).fill_random(1, 20 + i),
              ia.DeviceOperator(m, 1)) for i, m in enumerate(spaces)]
    calls = [(ALL_TERMS, PREC_FP64), (ALL_TERMS, PREC_MIXED), (ALL_TERMS & ~TERMS["comm222_pp_hhss"], PREC_FP64),
             (ALL_TERMS & ~TERMS["comm222_phss"], PREC_MIXED), (TERMS["comm222_phss"], PREC_MIXED),
             (ALL_TERMS & ~TERMS["comm221ss"], PREC_SPLIT), (ALL_TERMS & ~TERMS["comm122ss"], PREC_MIXED),
             (ALL_TERMS, PREC_FP64)]
    for mask, precision in calls:
        ia.Commutator.CommutatorScalarScalarBatched(pairs, mask, precision)
        got = [Z.to_host() for _, _, Z in pairs]
        for (X, Y, _), g in zip(pairs, got):
            ref = ia.Commutator.CommutatorScalarScalar(X, Y, mask, precision).to_host()
            assert g.herm == ref.herm and g.ZeroBody == ref.ZeroBody, (mask, precision)
            assert np.array_equal(g.OneBody, ref.OneBody) and np.array_equal(g.TwoBody, ref.TwoBody), (mask, precision)
