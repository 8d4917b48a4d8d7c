"""The FP32 pair functions that replace library calls (mixed precision):
r^alpha with 2 alpha an integer (roots and products), the ones beside them
that still call pow, and Helmholtz with and without damping, phases up to
three turns, in the neighbour-list walk and the cell rows, against the oracle
on the same grid or against FP64.

Bound: each FP32 pair term is within a few 6e-8 of its value; the sums of a
few hundred terms of either sign stay within 1e-6 of V and 1e-5 of the
gradient, the bounds of the mixed form elsewhere.  For r^3 the smooth part
dwarfs the pair terms and V's error is the FP32 grid's, which changes several
times over with the box alone (2.0e-7 to 6.7e-7 over the boxes here at 64^3), so
its bound is on the geometric mean over boxes, and a wider one on each.
Against the oracle wave numbers stay below a turn inside the cutoff, since the
matched polynomials cancel beyond; one source alone is taken to three turns.
(k0 = 2 has the same error as with library sines.)"""
import numpy as np
import pytest

from conftest import uniform_box

pytestmark = pytest.mark.gpu


def _run(oracle, kind, ko, coord, q, check=True, **kw):
    import npme_amd as N
    cx = kind == "Helmholtz"
    k = N.NPME_KeywordInput(calcType="pme", funcType=kind, EwaldSplit="DerivMatch", Rdir=6.0, BnOrder=6,
                            tol=1e-6, precision="mixed", N1=64, N2=64, N3=64, n1=16, n2=16, n3=16,
                            nDeriv=6, **kw)
    charge = {"chargeComplex": q} if cx else {"chargeReal": q}
    assert N.NPME_AddMissingKeywords(k, len(q), coord, **charge), N.npme_last_error()
    h = (N.NPME_Interface_SetUpComplexKernel if cx else N.NPME_Interface_SetUpRealKernel)(k, len(q), coord)
    assert h is not None, N.npme_last_error()
    m = oracle.compare_v(oracle.calcv(ko, (64, 64, 64), 6, coord, q), h.calcv(q))
    print(m["relV"], m["reldV"])
    if not check:
        return m
    assert m["relV"] < 1e-6 and m["reldV"] < 1e-5, m


@pytest.mark.parametrize("lists", ["on", "off"])
@pytest.mark.parametrize("alpha", [0.5, 1.5, -0.5, -2.5, 1.0, -2.0, -3.0, 0.3, -3.5])
def test_ralpha_pairs(oracle, alpha, lists):
    print("case ralpha pairs", alpha, lists, flush=True)
    coord, q = uniform_box(1500, 20.0)
    _run(oracle, "Ralpha", oracle.kernel(oracle.RALPHA, 6, 6.0, alpha=alpha), coord, q, alpha=alpha,
         neighborList=lists)


def test_ralpha_cubed(oracle):
    ms = []
    for seed, L in ((0, 20.0), (1, 27.3), (5, 30.0), (9, 31.7), (13, 34.1)):
        print("case r^3", seed, L, flush=True)
        coord, q = uniform_box(1500, L, seed, seed + 1) if seed else uniform_box(1500, L)
        ms.append(_run(oracle, "Ralpha", oracle.kernel(oracle.RALPHA, 6, 6.0, alpha=3.0), coord, q, check=False,
                       alpha=3.0))
    rel = {key: np.exp(np.mean(np.log([m[key] for m in ms]))) for key in ("relV", "reldV")}
    assert rel["relV"] < 1e-6 and rel["reldV"] < 1e-5, (rel, ms)


@pytest.mark.parametrize("lists", ["on", "off"])
@pytest.mark.parametrize("k0", [0.01, 0.5, 1.0, 1.1 + 0.2j, 0.3 + 0.01j])
def test_helmholtz_pairs(oracle, k0, lists):
    print("case helmholtz pairs", k0, lists, flush=True)
    coord, q = uniform_box(1500, 20.0)
    q = q + 1j * uniform_box(1500, 20.0, 7, 8)[1]
    k0 = complex(k0)
    _run(oracle, "Helmholtz", oracle.kernel(oracle.HELMHOLTZ, 6, 6.0, k0=k0), coord, q, k0_r=k0.real,
         k0_i=k0.imag, neighborList=lists)


@pytest.mark.parametrize("side", [20.0, 8.0])
@pytest.mark.parametrize("alpha", [0.5, 1.0, 3.0, -0.5, -2.0, 0.3])
def test_ralpha_coincident_charges(alpha, side):
    """Two charges at one place, in the cell rows and in dense cells: V is
    what the FP64 walk gives (r^alpha is 0 or infinite there, never NaN; 1e-5,
    ten times the mixed form's bound for a set), and the other charges' V and
    gradients are those of the list walk, which has the same grid part and the
    same pair terms summed in another order."""
    import npme_amd as N
    print("case coincident charges", alpha, side, flush=True)
    coord, q = uniform_box(1500, side)
    coord[11] = coord[10]
    V = {}
    for prec, lists in (("fp64", "off"), ("mixed", "off"), ("mixed", "on")):
        k = N.NPME_KeywordInput(calcType="pme", funcType="Ralpha", EwaldSplit="DerivMatch", Rdir=6.0, BnOrder=6,
                                tol=1e-6, precision=prec, N1=64, N2=64, N3=64, n1=16, n2=16, n3=16, nDeriv=6,
                                alpha=alpha, neighborList=lists)
        assert N.NPME_AddMissingKeywords(k, len(q), coord, chargeReal=q), N.npme_last_error()
        h = N.NPME_Interface_SetUpRealKernel(k, len(q), coord)
        assert h is not None, N.npme_last_error()
        assert ("neighbour list" if lists == "on" else "dense cells" if side == 8.0 else "cell rows") in h.Print()
        V[prec, lists] = h.calcv(q)
    at = np.array([10, 11])
    far = np.setdiff1d(np.arange(len(q)), at)
    a, b, c = V["mixed", "off"], V["fp64", "off"], V["mixed", "on"]
    rms = np.sqrt(np.mean(c[far, 0] ** 2))
    if alpha > 0:
        assert np.isfinite(a[at, 0]).all() and np.abs(a[at, 0] - b[at, 0]).max() < 1e-5 * rms, (a[at, 0], b[at, 0])
    else:
        assert np.array_equal(a[at, 0], b[at, 0]) and np.isinf(a[at, 0]).all(), (a[at, 0], b[at, 0])
    assert np.sqrt(np.mean((a[far, 0] - c[far, 0]) ** 2)) < 1e-6 * rms
    assert np.sqrt(np.mean((a[far, 1:] - c[far, 1:]) ** 2)) < 5e-6 * np.sqrt(np.mean(c[far, 1:] ** 2))


@pytest.mark.parametrize("lists", ["on", "off"])
@pytest.mark.parametrize("kw", [dict(alpha=a) for a in (0.5, 1.0, 2.5, 3.0, -0.5, -3.0, 0.3)] +
                         [dict(k0_r=k, k0_i=0.0) for k in (0.3, 1.0, 2.0, 3.0)] + [dict(k0_r=0.5, k0_i=0.1)])
def test_one_source(kw, lists):
    """One unit source, every target inside the cutoff: V is the pair function
    itself, mixed against FP64, phases to three turns.  Bound: the short-range
    part is the kernel less its matched polynomial, each rounded to FP32 a few
    times, so a few 6e-8 of S = |f| + sum |a_k| r^2k at the cutoff (for k0 = 3
    that sum is 1e3 times the kernel: hence the wide bounds of large phases),
    and for the grid part 1e-6 of the largest |V|, or for growing kernels 4e-7
    of the kernel across the grid's box, edges 2 (4 + 8): the FP32 transforms
    round by that scale (r^3: 9e3, where the pair itself is at most 216)."""
    import ctypes as C
    import npme_amd as N
    print("case one source", kw, lists, flush=True)
    cx = "k0_r" in kw
    kind, Rdir, Nder = ("Helmholtz" if cx else "Ralpha"), 6.0, 6
    rng = np.random.default_rng(4)
    coord = 4.0 + rng.uniform(-3.4, 3.4, (3000, 3))
    coord[0] = 4.0
    r = np.linalg.norm(coord - coord[0], axis=1)
    q = np.zeros(len(r), complex if cx else float)
    q[0] = 1.0
    V = {}
    for prec in ("mixed", "fp64"):
        k = N.NPME_KeywordInput(calcType="pme", funcType=kind, EwaldSplit="DerivMatch", Rdir=Rdir, BnOrder=6, tol=1e-6,
                                precision=prec, N1=64, N2=64, N3=64, n1=16, n2=16, n3=16, nDeriv=Nder,
                                neighborList=lists, **kw)
        assert N.NPME_AddMissingKeywords(k, len(q), coord, **({"chargeComplex": q} if cx else {"chargeReal": q}))
        h = (N.NPME_Interface_SetUpComplexKernel if cx else N.NPME_Interface_SetUpRealKernel)(k, len(q), coord)
        assert h is not None, N.npme_last_error()
        V[prec] = h.calcv(q)
    a, b = np.zeros((Nder + 1, 2)), np.zeros((Nder + 1, 2))
    assert N.lib().npme_dm_coefficients(kind.encode(), C.c_double(kw.get("alpha", 0.0)), C.c_double(kw.get("k0_r", 0.0)),
                                        C.c_double(kw.get("k0_i", 0.0)), C.c_int(Nder), C.c_double(Rdir),
                                        a.ctypes.data_as(C.c_void_p), b.ctypes.data_as(C.c_void_p)) == 0
    R2k = Rdir ** (2.0 * np.arange(Nder + 1))
    at = (r > 0.3) & (r < Rdir)
    f = np.abs(V["fp64"][at])
    S = [f[:, 0].max() + np.sum(np.hypot(*a.T) * R2k), f[:, 1:].max() + Rdir * np.sum(np.hypot(*b.T) * R2k)]
    d = np.abs(V["mixed"] - V["fp64"])[at]
    err = [d[:, 0].max(), d[:, 1:].max()]
    print("V %.2e of S, %.2e of max; gradient %.2e, %.2e" % (err[0] / S[0], err[0] / f[:, 0].max(), err[1] / S[1],
                                                             err[1] / f[:, 1:].max()))
    across = (12.0 * np.sqrt(3.0)) ** kw.get("alpha", -1.0)
    grid = [max(1e-6 * f[:, 0].max(), 4e-7 * across), max(1e-6 * f[:, 1:].max(), 4e-7 * across)]
    assert err[0] < 2.4e-7 * S[0] + grid[0] and err[1] < 2.4e-7 * S[1] + grid[1], (err, S, grid)


def test_ralpha_cubed_each_box():
    """r^3 box by box, against FP64 on the same grid: V within 2.4e-6, five
    times the rms of 300 boxes at 64^3 (4.8e-7; most of it the grid's k = 0
    term, a shift of V that is Gaussian over boxes), and without the shift
    within 1.4e-6, five times 2.8e-7."""
    import npme_amd as N
    for seed, L in ((0, 20.0), (1, 27.3), (5, 30.0), (9, 31.7), (13, 34.1), (21, 41.3)):
        print("case r^3 box", seed, L, flush=True)
        coord, q = uniform_box(1500, L, seed, seed + 1) if seed else uniform_box(1500, L)
        V = {}
        for prec in ("mixed", "fp64"):
            k = N.NPME_KeywordInput(calcType="pme", funcType="Ralpha", EwaldSplit="DerivMatch", Rdir=6.0, BnOrder=6,
                                    tol=1e-6, precision=prec, N1=64, N2=64, N3=64, n1=16, n2=16, n3=16, nDeriv=6,
                                    alpha=3.0)
            assert N.NPME_AddMissingKeywords(k, len(q), coord, chargeReal=q), N.npme_last_error()
            h = N.NPME_Interface_SetUpRealKernel(k, len(q), coord)
            assert h is not None, N.npme_last_error()
            V[prec] = h.calcv(q)[:, 0]
        d, norm = V["mixed"] - V["fp64"], np.linalg.norm(V["fp64"])
        print("%.2e %.2e" % (np.linalg.norm(d) / norm, np.linalg.norm(d - d.mean()) / norm))
        assert np.linalg.norm(d) < 2.4e-6 * norm and np.linalg.norm(d - d.mean()) < 1.4e-6 * norm
