"""One commutator with more 128x128 pp/hh tiles than two per CU: the first launch in two
parts (beside the pp/hh GEMM) or in one (without it) gives the same result."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


@pytest.mark.parametrize("small", [64, 0])
def test_first_launch_in_two_parts(ia, small):
    print(f"[gpu] first launch in two parts, small tiles up to {small}", flush=True)
    ms = ia.ModelSpace(9, "O16")  # 747 tiles, with the small channels on 128x128 tiles too more
    X = ia.DeviceOperator(ms, -1).fill_random(-1, 81)
    Y = ia.DeviceOperator(ms, 1).fill_random(1, 82)
    ref = None
    for overlap in (0, 1, 2):
        ms.set_tuning(overlap_pphh=overlap, pphh_small_tile_max=small)
        got = ia.Commutator.CommutatorScalarScalar(X, Y).to_host()
        ref = ref or got
        assert got.ZeroBody == ref.ZeroBody
        assert np.array_equal(got.OneBody, ref.OneBody) and np.array_equal(got.TwoBody, ref.TwoBody)
