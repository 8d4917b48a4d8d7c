"""The device set-up's sort by cell and its tile lists (scanned chunk by
chunk, or sorted) against the host set-up, which builds the same arrays with
a stable sort: the CalcV results are bit-identical only when every list holds
the same charges in the same order.

Sizes: fewer charges than a chunk of 64, a last chunk of one, several parts
per tile, cells longer than the ranking limit (2048, the radix sort's path),
enough tiles for the sorted lists, and many charges in few tiles (dozens of
parts a tile)."""
import time

import numpy as np
import pytest

from conftest import uniform_box

pytestmark = pytest.mark.gpu


def _calcv(coord, q, grid, prec, mode, Bn):
    import npme_amd as N
    k = N.NPME_KeywordInput(calcType="pme", funcType="Laplace", EwaldSplit="DerivMatch", Rdir=5.0, BnOrder=Bn,
                            tol=1e-6, precision=prec, N1=grid, N2=grid, N3=grid, n1=grid // 4, n2=grid // 4,
                            n3=grid // 4, nDeriv=6, setup=mode)
    assert N.NPME_AddMissingKeywords(k, len(q), coord, chargeReal=q), N.npme_last_error()
    h = N.NPME_Interface_SetUpRealKernel(k, len(q), coord)
    assert h is not None, N.npme_last_error()
    V = h.calcv(q)
    # and after a ResetCoord to mirrored positions, whose tables are the handle's own
    assert h.ResetCoord(len(q), coord.max(0) - coord), N.npme_last_error()
    return V, h.calcv(q)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("n,grid,Bn,packed", [(2, 40, 4, 0), (63, 40, 6, 0), (65, 48, 6, 0), (1000, 128, 8, 0),
                                              (6000, 64, 6, 4500), (140000, 512, 6, 0), (70001, 40, 6, 0),
                                              (70001, 128, 6, 5000)])
def test_device_lists_equal_host(n, grid, Bn, packed, prec):
    print("case set-up lists", n, grid, Bn, packed, prec, flush=True)
    side = max(14.0, (n / 0.1) ** (1.0 / 3.0))
    coord, q = uniform_box(n, side)
    if packed:  # most of the charges in one cell
        coord[:packed] = 0.5 * side + 0.02 * coord[:packed]
    dev = _calcv(coord, q, grid, prec, "device", Bn)
    host = _calcv(coord, q, grid, prec, "host", Bn)
    assert np.isfinite(dev[0]).all() and np.array_equal(dev[0], host[0])
    assert np.array_equal(dev[1], host[1])


def _reset_ms(coord, q, grid):
    """ResetCoord between two orders of the axes: the fastest of 10."""
    import npme_amd as N
    k = N.NPME_KeywordInput(calcType="pme", funcType="Laplace", EwaldSplit="DerivMatch", Rdir=4.0, BnOrder=6, tol=1e-6,
                            precision="mixed", N1=grid, N2=grid, N3=grid, n1=grid // 4, n2=grid // 4, n3=grid // 4,
                            nDeriv=6, neighborList="off")
    assert N.NPME_AddMissingKeywords(k, len(q), coord, chargeReal=q), N.npme_last_error()
    h = N.NPME_Interface_SetUpRealKernel(k, len(q), coord)
    assert h is not None, N.npme_last_error()
    sets, times = (coord[:, [1, 2, 0]].copy(), coord), []
    for i in range(12):
        t = time.perf_counter()
        assert h.ResetCoord(len(q), sets[i % 2]), N.npme_last_error()
        times.append(1e3 * (time.perf_counter() - t))
    return min(times[2:])


def test_few_tiles_cost():
    """A grid of 18 spreading tiles, whose lists are as long as the set: the
    tile scan shares them out over the chip, so the set-up costs what it does
    on a grid of 256 tiles (1.7 times that with 8 wavefronts a tile)."""
    print("case few tiles cost", flush=True)
    coord, q = uniform_box(1000000, 60.0)
    few, many = _reset_ms(coord, q, 40), _reset_ms(coord, q, 128)
    print(few, many)
    assert few < 1.15 * many


def test_crowded_cells_cost():
    """200,000 charges in a few dozen cells against the same number spread
    over the box: counting, ranking and block lists do not serialise on a
    crowded cell (3 times the time when they did)."""
    print("case crowded cells cost", flush=True)
    coord, q = uniform_box(200000, 60.0)
    spread = _reset_ms(coord, q, 96)
    coord[2:] = 31.0 + 0.03 * (coord[2:] - 30.0)
    coord[0], coord[1] = 0.0, 60.0
    crowded = _reset_ms(coord, q, 96)
    print(crowded, spread)
    assert crowded < 1.5 * spread
