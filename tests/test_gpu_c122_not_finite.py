"""comm122 with an Inf or NaN in an operand: it reaches the elements that are sums over it,
as in the oracle, and no others of its column bin (whole bins are multiplied at once)."""
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


def radial(nblk):
    """nblk radial states of l = 0 and of l = 1, j = 1/2: groups of up to nblk^2 kets."""
    n, l, j2, tz2, occ, cvq = [], [], [], [], [], []
    for r in range(nblk):
        for ll in (0, 1):
            for t in (-1, 1):
                core = r == 0 and ll == 0
                n.append(r); l.append(ll); j2.append(1); tz2.append(t)
                occ.append(1.0 if core else 0.0)
                cvq.append(0 if core else 2)
    return dict(n=n, l=l, j2=j2, tz2=tz2, occ=occ, cvq=cvq)


@pytest.mark.parametrize("basis", ["emax4", "emax7", "radial4", "radial9"])
@pytest.mark.parametrize("which", ["X", "Y"])
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_comm122_not_finite(ia, basis, which, value):
    print(f"[gpu] comm122 {value} in {which}, {basis}", flush=True)
    if basis.startswith("emax"):
        ms, orc = ia.ModelSpace(int(basis[4:]), "O16"), OracleModelSpace(int(basis[4:]), 16, 8)
    else:
        orb = radial(int(basis[6:]))
        ms, orc = ia.ModelSpace(2, orbits=orb), OracleModelSpace(2, orbits=orb)
    ops = {"X": random_op(orc, -1, 61), "Y": random_op(orc, 1, 62)}
    bad = ops[which]
    ch = max(ms.channels, key=lambda c: c["n"])
    n, off = ch["n"], ch["off"]
    for r, c in ((1, n // 2), (n - 1, n // 3)):
        bad["two"][off + c * n + r] = value
        bad["two"][off + r * n + c] = bad["herm"] * value
    dX = ia.Operator(ms, -1, 0.0, ops["X"]["one"], ops["X"]["two"]).to_device()
    dY = ia.Operator(ms, 1, 0.0, ops["Y"]["one"], ops["Y"]["two"]).to_device()
    Z = np.asarray(ia.Commutator.CommutatorScalarScalar(dX, dY, TERMS["comm122ss"]).to_host().TwoBody)
    R = orc.commutator(ops["X"], ops["Y"], TERMS["comm122ss"])["two"]
    good = np.isfinite(R)
    assert 0 < np.count_nonzero(~good) < 40 * n  # a few rows and columns of one channel at most
    assert np.array_equal(np.isfinite(Z), good)
    assert np.max(np.abs(Z[good] - R[good])) <= TOL * np.max(np.abs(R[good]))
