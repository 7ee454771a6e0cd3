"""The one-pass kernels that sum an operator's norm (alone, with a copy, with an axpy) on
channel blocks of every alignment, from an empty two-body part to many chunks.

Tolerance: the kernel adds at most 8 + 8 terms per thread, 6 + 2 levels of a tree per
block and 8 + 8 over the blocks, all positive, so the sums are within 48 * 2^-53 < 6e-15
of the exact ones (longdouble here) and the norms within 3e-15."""
import numpy as np
import pytest

from opgen import random_op

pytestmark = pytest.mark.gpu
TOL = 1e-14


@pytest.fixture(scope="module")
def ia():
    import imsrg_amd
    return imsrg_amd


def norms(ms, op):
    one = sum(np.longdouble(ms.orbits[i]["j2"] + 1) * np.sum(op.OneBody[i].astype(np.longdouble) ** 2)
              for i in range(ms.norb))
    two = np.longdouble(0)
    for c in ms.channels:
        v = op.TwoBody[c["off"]:c["off"] + c["n"] ** 2].astype(np.longdouble)
        two += (2 * c["J"] + 1) ** 2 * np.sum(v * v)
    return float(np.sqrt(one)), float(np.sqrt(two))


@pytest.mark.parametrize("emax,ref", [(0, "He4"), (1, "O16"), (2, "O16"), (3, "O18"), (4, "O16"), (6, "O16")])
def test_norm_copy_axpy(ia, emax, ref):
    print(f"[gpu] norm pass emax={emax} {ref}", flush=True)
    ms = ia.ModelSpace(emax, ref)
    r = random_op(ms, 1, 77 + emax)
    h = ia.Operator(ms, 1, 0.25, r["one"], r["two"])
    d = h.to_device()
    n1, n2 = norms(ms, h)
    g1, g2, g = d.norms()
    assert abs(g1 - n1) <= TOL * n1 and abs(g2 - n2) <= TOL * max(n2, 1.0)
    assert abs(g - np.hypot(n1, n2)) <= TOL * np.hypot(n1, n2)
    # the copy inside normal ordering: the two-body part comes over bit for bit
    out = ia.DeviceOperator(ms, 1)
    out.fill_random(1, 5)
    d.DoNormalOrdering(out=out)
    assert np.array_equal(out.to_host().TwoBody, h.TwoBody)
    # the axpy inside BCH_Transform: with one term, Out = Op + [Omega, Op]
    w = random_op(ms, -1, 99 + emax, scale1=0.1, scale2=0.1)
    W = ia.Operator(ms, -1, 0.0, w["one"], w["two"]).to_device()
    try:
        ia.BCH.BCH_Transform(d, W, out=out, max_terms=1)
    except ia.HipError:
        pass  # one term does not converge; Out holds it all the same
    z = ia.Commutator.CommutatorScalarScalar(W, d).to_host()
    got = out.to_host()
    assert np.array_equal(got.TwoBody, h.TwoBody + z.TwoBody)
    assert np.array_equal(got.OneBody, h.OneBody + z.OneBody)
    assert got.ZeroBody == h.ZeroBody + z.ZeroBody
