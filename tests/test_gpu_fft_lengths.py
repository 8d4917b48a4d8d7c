"""The general FFT passes at lengths that use every radix (2 to 10, 12, 16;
2 only at 8 to 32) and two, three and four stages, to the longest lengths
(4092 at most), on each of the three axes: CalcV on a given
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


# with a spline of order 4: 20 = 10 2, 24 = 12 2, 32 = 16 2
SHORT = [(20, 24, 32), (32, 20, 24), (24, 32, 20)]
# one column to a workgroup in FP64 (rows of more than half its LDS), the
# largest workgroups and index quotients: 3840 = 10 8 8 6, 4032 = 8 9 8 7,
# 4000 = 10 10 8 5, 2592 = 8 9 6 6, 3888 = 8 9 9 6
LONG = [(36, 40, 3840), (4032, 36, 40), (36, 4000, 40), (2592, 36, 40), (40, 3888, 36), (36, 40, 4032)]


def _setup(kind, prec, grid, coord, Bn=6):
    import npme_amd as N
    kw = dict(calcType="pme", EwaldSplit="DerivMatch", Rdir=6.0, BnOrder=Bn, tol=1e-6, precision=prec,
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


def _cases():
    return [(g, 4) for g in SHORT] + [(g, 6) for g in LONG]


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["Laplace", "Helmholtz"])
@pytest.mark.parametrize("grid,Bn", _cases())
def test_fft_shortest_and_longest_lengths(oracle, grid, Bn, kind, prec):
    print("case fft lengths", grid, Bn, kind, prec, flush=True)
    coord, q = uniform_box(401, 20.0)
    if kind == "Helmholtz":
        q = q + 1j * uniform_box(401, 20.0, 7, 8)[1]
    V = _setup(kind, prec, grid, coord, Bn).calcv(q)
    k = oracle.kernel(oracle.LAPLACE, 6, 6.0) if kind == "Laplace" else \
        oracle.kernel(oracle.HELMHOLTZ, 6, 6.0, k0=0.5)
    m = oracle.compare_v(oracle.calcv(k, grid, Bn, coord, q), V)
    print(m["relV"], m["reldV"])
    bound = (1e-11, 1e-11) if prec == "fp64" else (1e-6, 1e-5)
    assert m["relV"] < bound[0] and m["reldV"] < bound[1], m


@pytest.mark.parametrize("grid,bound", [(48, 1.57e-7), (96, 1.61e-7), (144, 1.62e-7)])
def test_radix16_rounding(grid, bound):
    """FP32 rounding of grids whose transforms have a radix 16 stage: mixed
    against FP64, mean over 24 boxes of the error of V without its mean (the
    k = 0 term, which varies several times over from box to box).  The
    constants of that stage rounded to FP32 gave 1.70e-7, 1.77e-7 and 1.82e-7,
    radices up to 8 1.74e-7, 1.76e-7 and 1.79e-7; with their low parts it is
    1.43e-7, 1.46e-7 and 1.43e-7.  The bounds lie halfway."""
    import npme_amd as N
    print("case radix 16 rounding", grid, flush=True)
    errs = []
    for b in range(24):
        coord, q = uniform_box(500, 26.0 + 0.3 * b, 11 + 4 * b, 12 + 4 * b)
        V = {}
        for prec in ("mixed", "fp64"):
            k = N.NPME_KeywordInput(calcType="pme", funcType="Laplace", EwaldSplit="DerivMatch", Rdir=6.0, BnOrder=6,
                                    tol=1e-6, precision=prec, N1=grid, N2=grid, N3=grid, n1=grid // 4, n2=grid // 4,
                                    n3=grid // 4, nDeriv=6)
            assert N.NPME_AddMissingKeywords(k, len(q), coord, chargeReal=q), N.npme_last_error()
            h = N.NPME_Interface_SetUpRealKernel(k, len(q), coord)
            assert h is not None, N.npme_last_error()
            V[prec] = h.calcv(q)[:, 0]
        d = V["mixed"] - V["fp64"]
        errs.append(np.linalg.norm(d - d.mean()) / np.linalg.norm(V["fp64"]))
    print("%.3e" % np.mean(errs))
    assert np.mean(errs) < bound, errs
