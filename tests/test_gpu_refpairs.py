"""The direct sum over the reference's interacting cell pairs (erfc split) by
wavefronts of a few targets of one cell, and by a thread per target for stencils wider than
nNeigh = 3: cells of 0 to 9 charges (batches of 4 targets, chunks of 64
candidates) and one packed with hundreds, against the oracle's pair set.

Bound: FP64 1e-11, the sums' rounding through the potential's cancellation."""
import re

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


def test_refpairs_crowded_cell(oracle):
    """Nearly all charges in one cell: its targets are shared out (at most 8 a
    wavefront), so a crowded cell does not hold up the launch (2,500 charges in
    one cell on a single wavefront: 42 ms against 3.3 ms on 40)."""
    import npme_amd as N
    n = 2003
    print("case refpairs crowded", n, flush=True)
    coord, q = uniform_box(n, 22.0)
    coord[:n - 60] = 9.1 + 0.08 * coord[:n - 60]  # inside the cell [9, 12)
    coord[n - 2], coord[n - 1] = 0.0, 22.0
    k = N.NPME_KeywordInput(calcType="pme", funcType="Laplace", EwaldSplit="LaplaceOrig", Rdir=6.0, BnOrder=6,
                            tol=1e-6, precision="fp64", N1=64, N2=64, N3=64, n1=16, n2=16, n3=16, nNeigh=2,
                            nCellClust1D=3, nDeriv=6)
    assert N.NPME_AddMissingKeywords(k, n, coord, chargeReal=q), N.npme_last_error()
    for mode in ("device", "host"):
        k.AddKeyword("setup", mode)
        h = N.NPME_Interface_SetUpRealKernel(k, n, coord)
        assert h is not None, N.npme_last_error()
        V = h.calcv(q)
        ko = oracle.kernel_erf(6.0, oracle.rdir2beta(6.0, 1e-6))
        m = oracle.compare_v(oracle.calcv_laplace_orig(ko, (64, 64, 64), 6, coord, q, nNeigh=2, nCellClust1D=3), V)
        print(m["relV"], m["reldV"])
        assert m["relV"] < 1e-11 and m["reldV"] < 1e-11, m
        wavefronts = re.search(r"every point pair \(FP64\), (\d+) wavefronts", h.Print())
        assert wavefronts and (n - 60) / 8 <= int(wavefronts.group(1)) <= n / 8 + 61, h.Print()
