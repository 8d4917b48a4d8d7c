"""The general FFT passes at lengths that use every radix (2 to 10, 12, 16)
and two, three and four stages, on each of the three axes: CalcV on a given
grid against the oracle on the same grid.  Real charges (R2C and C2R rows,
columns, convolution) and complex ones (complex rows), FP64 and mixed.

Bounds: FP64 1e-11, the transforms' rounding (1e-16 log2 N) times the
cancellation of the potential; mixed 1e-6 in V and 1e-5 in its gradient,
FP32 rounding of the grid (6e-8) through the same."""
import numpy as np
import pytest

from conftest import uniform_box

pytestmark = pytest.mark.gpu

# (N1, N2, N3): 1372 = 7 7 7 4, 980 = 4 7 7 5, 1260 = 4 stages, 36 = 12 3,
# 40 = 10 4, 64 = 16 4, 100 = 10 10, 108 = 12 9, 112 = 16 7, 140 = 4 7 5,
# 144 = 16 9, 48 = 16 3, 160 = 16 10, 280 = 8 7 5, 540 = 3 stages
GRIDS = [(36, 40, 48), (64, 56, 60), (100, 108, 112), (144, 140, 160), (280, 36, 72),
         (36, 540, 40), (40, 36, 500), (980, 36, 40), (36, 1372, 40), (40, 36, 1260)]


def _setup(kind, prec, grid, coord):
    import npme_amd as N
    kw = dict(calcType="pme", EwaldSplit="DerivMatch", Rdir=6.0, BnOrder=6, tol=1e-6, precision=prec,
              nDeriv=6, fftKernels="generic")
    kw.update({"N%d" % (d + 1): n for d, n in enumerate(grid)})
    kw.update({"n%d" % (d + 1): n // 4 for d, n in enumerate(grid)})
    if kind == "Helmholtz":
        kw.update(k0_r=0.5, k0_i=0.0)
    k = N.NPME_KeywordInput(funcType=kind, **kw)
    q = {"chargeReal": np.ones(len(coord))} if kind == "Laplace" else {"chargeComplex": np.ones(len(coord), complex)}
    assert N.NPME_AddMissingKeywords(k, len(coord), coord, **q), N.npme_last_error()
    f = N.NPME_Interface_SetUpRealKernel if kind == "Laplace" else N.NPME_Interface_SetUpComplexKernel
    h = f(k, len(coord), coord)
    assert h is not None, N.npme_last_error()
    assert (h.Get_N1(), h.Get_N2(), h.Get_N3()) == grid
    return h


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["Laplace", "Helmholtz"])
@pytest.mark.parametrize("grid", GRIDS)
def test_fft_lengths_match_oracle(oracle, grid, kind, prec):
    print("case fft lengths", grid, kind, prec, flush=True)
    coord, q = uniform_box(401, 20.0)
    if kind == "Helmholtz":
        q = q + 1j * uniform_box(401, 20.0, 7, 8)[1]
    V = _setup(kind, prec, grid, coord).calcv(q)
    k = oracle.kernel(oracle.LAPLACE, 6, 6.0) if kind == "Laplace" else \
        oracle.kernel(oracle.HELMHOLTZ, 6, 6.0, k0=0.5)
    m = oracle.compare_v(oracle.calcv(k, grid, 6, coord, q), V)
    print(m["relV"], m["reldV"])
    bound = (1e-11, 1e-11) if prec == "fp64" else (1e-6, 1e-5)
    assert m["relV"] < bound[0] and m["reldV"] < bound[1], m
