"""Small grids: several wavefronts share a spreading tile (1, 2 or 4 by the
tiles and the length of their lists) and interpolation tiles shrink (edges 4
to 16).  Charge counts around a chunk of 64 and its multiples, spread over the
box or packed into one corner of it, against the oracle on the same grid.

Bounds: FP64 1e-11 and mixed 1e-6 / 1e-5, as for the same kernels elsewhere:
the wavefronts' partial sums are added in FP64.  (At least 40 charges: of two
charges 10 apart V is 0.06 of the self terms it is left over from, so FP32
rounding of those terms, 6e-8 each, already shows as 1e-6 of V.)"""
import numpy as np
import pytest

from conftest import uniform_box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["Laplace", "Helmholtz"])
@pytest.mark.parametrize("n,grid,Bn,packed", [(40, 40, 6, False), (64, 40, 6, False), (65, 40, 4, True),
                                              (700, 40, 6, False), (2100, 40, 8, False), (2100, 64, 12, True),
                                              (1500, 128, 6, True), (900, 160, 10, False)])
def test_few_tiles_match_oracle(oracle, n, grid, Bn, packed, kind, prec):
    import npme_amd as N
    print("case few tiles", n, grid, Bn, packed, kind, prec, flush=True)
    coord, q = uniform_box(n, 16.0)
    if packed:  # all but two corners of the box into an eighth of its edge
        coord[2:] *= 0.125
        coord[0], coord[1] = 0.0, 16.0
    cx = kind == "Helmholtz"
    if cx:
        q = q + 1j * uniform_box(n, 16.0, 7, 8)[1]
    kw = dict(k0_r=0.5, k0_i=0.0) if cx else {}
    k = N.NPME_KeywordInput(calcType="pme", funcType=kind, EwaldSplit="DerivMatch", Rdir=5.0, BnOrder=Bn,
                            tol=1e-6, precision=prec, N1=grid, N2=grid, N3=grid, n1=grid // 4, n2=grid // 4,
                            n3=grid // 4, nDeriv=6, **kw)
    assert N.NPME_AddMissingKeywords(k, n, coord, **({"chargeComplex": q} if cx else {"chargeReal": q})), \
        N.npme_last_error()
    h = (N.NPME_Interface_SetUpComplexKernel if cx else N.NPME_Interface_SetUpRealKernel)(k, n, coord)
    assert h is not None, N.npme_last_error()
    V = h.calcv(q)
    assert np.array_equal(V, h.calcv(q))  # the order of the sums is fixed
    ko = oracle.kernel(oracle.HELMHOLTZ, 6, 5.0, k0=0.5) if cx else oracle.kernel(oracle.LAPLACE, 6, 5.0)
    m = oracle.compare_v(oracle.calcv(ko, (grid,) * 3, Bn, coord, q), V)
    print(m["relV"], m["reldV"])
    bound = (1e-11, 1e-11) if prec == "fp64" else (1e-6, 1e-5)
    assert m["relV"] < bound[0] and m["reldV"] < bound[1], m


def _interp_us(n, packed):
    """Interpolation stage of a set of n charges on a 64^3 grid: the fastest of
    40 calls (device time between events)."""
    import npme_amd as N
    coord, q = uniform_box(n, 32.0)
    if packed:
        coord[2:] = 16.0 + 0.06 * (coord[2:] - 16.0)
        coord[0], coord[1] = 0.0, 32.0
    k = N.NPME_KeywordInput(calcType="pme", funcType="Laplace", EwaldSplit="DerivMatch", Rdir=5.0, BnOrder=6, tol=1e-6,
                            precision="mixed", N1=64, N2=64, N3=64, n1=16, n2=16, n3=16, nDeriv=6)
    assert N.NPME_AddMissingKeywords(k, n, coord, chargeReal=q), N.npme_last_error()
    h = N.NPME_Interface_SetUpRealKernel(k, n, coord)
    assert h is not None, N.npme_last_error()
    h.set_profiling(True)
    times = []
    for _ in range(40):
        h.calcv(q)
        times.append(h.stage_times()[-1])
    return 1e3 * min(times)


def test_crowded_interpolation_tile():
    """6,000 charges that fall into a few tiles of edge 4: their tile must
    have a whole block of wavefronts.  About 8 times the time of the same
    number spread out, and 24 times with one wavefront a tile: bound 14."""
    print("case crowded tile", flush=True)
    spread, packed = _interp_us(6000, False), _interp_us(6000, True)
    print(spread, packed)
    assert packed < 14 * spread
