"""Every phase of a profiled commutator has its time, on bases whose commutators otherwise
put several phases into one launch too, and the result is the same bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


@pytest.mark.parametrize("emax", [2, 4, 7])
@pytest.mark.parametrize("precision", [0, 1, 2])
def test_every_phase_is_timed(ia, emax, precision):
    print(f"[gpu] phase times emax={emax} precision={precision}", flush=True)
    ms = ia.ModelSpace(emax, "O16")
    X = ia.DeviceOperator(ms, -1).fill_random(-1, 51)
    Y = ia.DeviceOperator(ms, 1).fill_random(1, 52)
    ref = ia.Commutator.CommutatorScalarScalar(X, Y, precision=precision).to_host()
    default = ms.get_tuning()["overlap_pphh"]
    try:
        for overlap in (0, 1, 2):
            ms.set_tuning(overlap_pphh=overlap)
            ms.set_profiling(True)
            ms.phase_times()
            got = ia.Commutator.CommutatorScalarScalar(X, Y, precision=precision).to_host()
            assert min(ms.phase_times()) > 0.0, overlap
            ms.set_profiling(False)
            assert got.ZeroBody == ref.ZeroBody
            assert np.array_equal(got.OneBody, ref.OneBody) and np.array_equal(got.TwoBody, ref.TwoBody)
    finally:
        ms.set_profiling(False)
        ms.set_tuning(overlap_pphh=default)
