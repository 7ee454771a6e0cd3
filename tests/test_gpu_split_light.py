"""Split products with a light reference, whose pp/hh GEMM is placed before the first launch:
the same result as on one stream, eagerly, profiled and replayed as a graph."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


def test_split_products_light_reference(ia):
    print("[gpu] split products, emax=7 He4", flush=True)
    ms = ia.ModelSpace(7, "He4")
    X = ia.DeviceOperator(ms, -1).fill_random(-1, 61)
    Y = ia.DeviceOperator(ms, 1).fill_random(1, 62)
    Z = ia.DeviceOperator(ms, 1)

    def same(mask):
        got = ia.Commutator.CommutatorScalarScalar(X, Y, mask, ia.PREC_SPLIT, out=Z).to_host()
        ref = refs[mask]
        assert got.ZeroBody == ref.ZeroBody
        assert np.array_equal(got.OneBody, ref.OneBody) and np.array_equal(got.TwoBody, ref.TwoBody)

    masks = (ia.ALL_TERMS, ia.ALL_TERMS & ~ia.TERMS["comm222_phss"], ia.TERMS["comm222_pp_hhss"])
    default = ms.get_tuning()["overlap_pphh"]
    try:
        ms.set_tuning(overlap_pphh=0)
        refs = {m: ia.Commutator.CommutatorScalarScalar(X, Y, m, ia.PREC_SPLIT).to_host() for m in masks}
        ms.set_tuning(overlap_pphh=1)
        for m in masks:
            same(m)
        ms.set_profiling(True)
        same(ia.ALL_TERMS)
        assert min(ms.phase_times()) > 0.0
        ms.set_profiling(False)
        ms.set_graphs(True)
        for _ in range(3):
            same(ia.ALL_TERMS)
            Y.axpy(0.0, X)  # eager work between the replays
            ms.synchronize()
    finally:
        ms.set_graphs(False)
        ms.set_profiling(False)
        ms.set_tuning(overlap_pphh=default)
