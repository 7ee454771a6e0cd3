"""Batched commutators on operands that change from call to call: the batch keeps its
work lists per contexts, and each call writes its operands into the device table in
groups of 64 pairs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


@pytest.mark.parametrize("npairs", [1, 2, 64, 65])
def test_batch_follows_its_operands(ia, npairs):
    print(f"[gpu] batch operands npairs={npairs}", flush=True)
    spaces = [ia.ModelSpace(2, "O16"), ia.ModelSpace(1, "He4")]
    ms = [spaces[i % 2] for i in range(npairs)]

    def pairs(seed, hx, hy):
        return [(ia.DeviceOperator(m, hx).fill_random(hx, seed + 2 * i),
                 ia.DeviceOperator(m, hy).fill_random(hy, seed + 2 * i + 1), ia.DeviceOperator(m, 1))
                for i, m in enumerate(ms)]

    # other operands, other Hermiticities and the first operands again, with no
    # synchronisation between the calls
    sets = [pairs(100, -1, 1), pairs(1000, 1, 1), pairs(2000, -1, -1)]
    for s in (0, 1, 2, 0):
        ia.Commutator.CommutatorScalarScalarBatched(sets[s])
    for s in sets:
        for X, Y, Z in s:
            got = Z.to_host()
            ref = ia.Commutator.CommutatorScalarScalar(X, Y).to_host()
            assert got.herm == ref.herm and got.ZeroBody == ref.ZeroBody
            assert np.array_equal(got.OneBody, ref.OneBody) and np.array_equal(got.TwoBody, ref.TwoBody)
