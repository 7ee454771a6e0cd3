"""What BCH_Transform and BCH_Product leave in their result operator: nothing new when an
operand holds Inf or NaN, the same bits in place as beside the operand, and the operand
itself when no term is needed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


def state(d):
    o = d.to_host()
    return o.herm, o.ZeroBody, o.OneBody.tobytes(), o.TwoBody.tobytes()


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("where", ["first", "second"])
def test_out_untouched_when_not_finite(ia, value, where):
    print(f"[gpu] bch out, {where} operand {value}", flush=True)
    ms = ia.ModelSpace(2, "O16")
    bad = ia.DeviceOperator(ms, -1).fill_random(-1, 5).to_host()
    i, j = next((i, j) for i in range(ms.norb) for j in range(i) if bad.OneBody[i, j] != 0.0)
    bad.OneBody[i, j], bad.OneBody[j, i] = value, -value
    bad, good = bad.to_device(), ia.DeviceOperator(ms, -1).fill_random(-1, 6)
    ops = (bad, good) if where == "first" else (good, bad)
    out = ia.DeviceOperator(ms, 1).fill_random(1, 7)
    before = state(out)
    for call in (ia.BCH.BCH_Transform, ia.BCH.BCH_Product):
        with pytest.raises(ia.HipError):
            call(*ops, out=out)
        assert state(out) == before


@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("precision", [0, 1])
def test_transform_in_place(ia, graphs, precision):
    print(f"[gpu] bch in place graphs={graphs} precision={precision}", flush=True)
    ms = ia.ModelSpace(4, "O16")
    W = ia.DeviceOperator(ms, -1).fill_random(-1, 11)
    W.scale(0.02)
    H = ia.DeviceOperator(ms, 1).fill_random(1, 12)
    ref = state(ia.BCH.BCH_Transform(H, W, precision=precision))
    try:
        ms.set_graphs(graphs)
        op = ia.DeviceOperator(ms, 1)
        for _ in range(3):
            op.copy_from(H)
            ia.BCH.BCH_Transform(op, W, out=op, precision=precision)
            assert state(op) == ref
    finally:
        ms.set_graphs(False)


def test_transform_without_terms(ia):
    print("[gpu] bch without terms", flush=True)
    ms = ia.ModelSpace(2, "O16")
    W = ia.DeviceOperator(ms, -1).fill_random(-1, 21)
    H = ia.DeviceOperator(ms, 1).fill_random(1, 22)
    H.scale(1e-14)
    out = ia.DeviceOperator(ms, -1).fill_random(-1, 23)
    ia.BCH.BCH_Transform(H, W, out=out)
    assert state(out) == state(H)
