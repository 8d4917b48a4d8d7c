"""The direct sum over the reference's interacting cell pairs (erfc split) by
a wavefront per cell, and by a thread per target for stencils wider than
nNeigh = 3: cells of 0 to 9 charges (batches of 4 targets, chunks of 64
candidates) and one packed with hundreds, against the oracle's pair set.

Bound: FP64 1e-11, the sums' rounding through the potential's cancellation."""
import numpy as np
import pytest

from conftest import uniform_box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("packed", [0, 300])
@pytest.mark.parametrize("nNeigh,nClust", [(1, 3), (2, 3), (3, 3), (4, 5)])
def test_refpairs_match_oracle(oracle, nNeigh, nClust, packed):
    import npme_amd as N
    print("case refpairs", nNeigh, nClust, packed, flush=True)
    coord, q = uniform_box(1201, 22.0)
    if packed:
        coord[:packed] = 9.0 + 0.06 * coord[:packed]
    k = N.NPME_KeywordInput(calcType="pme", funcType="Laplace", EwaldSplit="LaplaceOrig", Rdir=6.0, BnOrder=6,
                            tol=1e-6, precision="fp64", N1=64, N2=64, N3=64, n1=16, n2=16, n3=16,
                            nNeigh=nNeigh, nCellClust1D=nClust, nDeriv=6)
    assert N.NPME_AddMissingKeywords(k, len(q), coord, chargeReal=q), N.npme_last_error()
    h = N.NPME_Interface_SetUpRealKernel(k, len(q), coord)
    assert h is not None, N.npme_last_error()
    V = h.calcv(q)
    assert np.array_equal(V, h.calcv(q)) and np.array_equal(V, h.calcv(q))  # graph replays
    ko = oracle.kernel_erf(6.0, oracle.rdir2beta(6.0, 1e-6))
    m = oracle.compare_v(oracle.calcv_laplace_orig(ko, (64, 64, 64), 6, coord, q, nNeigh=nNeigh,
                                                   nCellClust1D=nClust), V)
    print(m["relV"], m["reldV"])
    assert m["relV"] < 1e-11 and m["reldV"] < 1e-11, m
