"""comm122 against the oracle where its column bins change shape: one-body blocks of
many orbits (groups of kets past one 16-column block, past 64 columns), and channels of
fewer rows than a wave takes."""
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


@pytest.mark.parametrize("nblk", [1, 3, 4, 5, 6, 8, 9, 12])
def test_comm122_block_sizes(ia, nblk):
    # nblk radial states of l = 0 and of l = 1, j = 1/2: groups of up to nblk^2 kets
    print(f"[gpu] comm122 bins nblk={nblk}", flush=True)
    n, l, j2, tz2, occ, cvq = [], [], [], [], [], []
    for r in range(nblk):
        for ll in (0, 1):
            for t in (-1, 1):
                n.append(r); l.append(ll); j2.append(1); tz2.append(t)
                occ.append(1.0 if r == 0 and ll == 0 else 0.0)
                cvq.append(0 if r == 0 and ll == 0 else 2)
    orb = dict(n=n, l=l, j2=j2, tz2=tz2, occ=occ, cvq=cvq)
    ms, orc = ia.ModelSpace(2, orbits=orb), OracleModelSpace(2, orbits=orb)
    for hx, hy in ((-1, 1), (1, 1)):
        X, Y = random_op(orc, hx, 11 + nblk), random_op(orc, hy, 31 + nblk)
        dX = ia.Operator(ms, hx, 0.0, X["one"], X["two"]).to_device()
        dY = ia.Operator(ms, hy, 0.0, Y["one"], Y["two"]).to_device()
        Z = ia.Commutator.CommutatorScalarScalar(dX, dY, TERMS["comm122ss"]).to_host()
        R = orc.commutator(X, Y, TERMS["comm122ss"])
        assert np.max(np.abs(Z.TwoBody - R["two"])) <= TOL * max(np.max(np.abs(R["two"])), 1e-300)
