"""The direct sum of densely packed charges (blocks of 64 targets and groups
of 16 sources of one cell, k_direct_fine) against the oracle and against the
cell-row walk (which the host set-up takes), for every kernel in both
precisions: packed balls
with cells of hundreds of charges, partial blocks and groups, stray charges
alone in their cells, near-coincident pairs (the fixed point's residuals), a
cluster of one cell per axis and stencils of nNeigh 1 to 3.

Bounds: FP64 1e-11.  Mixed against the cell rows, which sum the same pair
terms in another order: 1e-6 of V and 5e-6 of the gradient."""
import numpy as np
import pytest

from conftest import uniform_box

pytestmark = pytest.mark.gpu


def _charges(n, cx):
    coord, q = uniform_box(n, 1.0)
    rng = np.random.default_rng(5)
    ball = rng.standard_normal((n, 3)) * 0.8 + np.where(np.arange(n)[:, None] % 3 == 0, 4.0, 11.0)
    coord = np.where(np.arange(n)[:, None] < 7, 18.0 * coord, ball)
    coord[20:23] = coord[30:33] + 1e-3 * (1 + np.arange(3))[:, None]
    return coord, (q + 1j * uniform_box(n, 1.0, 7, 8)[1] if cx else q)


def _setup(kind, prec, coord, q, mode, nNeigh, nClust, **kw):
    import npme_amd as N
    cx = kind == "Helmholtz"
    k = N.NPME_KeywordInput(calcType="pme", funcType=kind, EwaldSplit="DerivMatch", Rdir=4.0, BnOrder=6, tol=1e-6,
                            precision=prec, N1=96, N2=96, N3=96, n1=24, n2=24, n3=24, nDeriv=6, nNeigh=nNeigh,
                            nCellClust1D=nClust, neighborList="off", setup=mode, **kw)
    assert N.NPME_AddMissingKeywords(k, len(q), coord, **({"chargeComplex": q} if cx else {"chargeReal": q})), \
        N.npme_last_error()
    h = (N.NPME_Interface_SetUpComplexKernel if cx else N.NPME_Interface_SetUpRealKernel)(k, len(q), coord)
    assert h is not None, N.npme_last_error()
    return h


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind,kw", [("Laplace", {}), ("Ralpha", {"alpha": -1.5}), ("Ralpha", {"alpha": -0.3}),
                                     ("Helmholtz", {"k0_r": 0.5, "k0_i": 0.0}),
                                     ("Helmholtz", {"k0_r": 0.5, "k0_i": 0.1})])
@pytest.mark.parametrize("nNeigh,nClust", [(1, 2), (2, 3), (3, 3)])
def test_dense_cells(oracle, nNeigh, nClust, kind, kw, prec):
    print("case dense cells", nNeigh, nClust, kind, kw, prec, flush=True)
    coord, q = _charges(8009, kind == "Helmholtz")
    h = _setup(kind, prec, coord, q, "device", nNeigh, nClust, **kw)
    dense = "dense cells" in h.Print()
    V = h.calcv(q)
    assert np.array_equal(V, h.calcv(q)) and np.array_equal(V, h.calcv(q))  # graph replays
    Vr = _setup(kind, prec, coord, q, "host", nNeigh, nClust, **kw).calcv(q)
    d = V - Vr
    rel = np.sqrt(np.mean(np.abs(d[:, 0]) ** 2)) / np.sqrt(np.mean(np.abs(Vr[:, 0]) ** 2))
    relg = np.sqrt(np.mean(np.abs(d[:, 1:]) ** 2)) / np.sqrt(np.mean(np.abs(Vr[:, 1:]) ** 2))
    print(dense, rel, relg)
    assert dense
    if prec == "mixed":
        assert rel < 1e-6 and relg < 5e-6
        return
    assert rel < 1e-11 and relg < 1e-11
    ok = {"Laplace": lambda: oracle.kernel(oracle.LAPLACE, 6, 4.0),
          "Ralpha": lambda: oracle.kernel(oracle.RALPHA, 6, 4.0, alpha=kw.get("alpha", 0.0)),
          "Helmholtz": lambda: oracle.kernel(oracle.HELMHOLTZ, 6, 4.0,
                                             k0=complex(kw.get("k0_r", 0.0), kw.get("k0_i", 0.0)))}[kind]()
    m = oracle.compare_v(oracle.calcv(ok, (96, 96, 96), 6, coord, q), V)
    print(m["relV"], m["reldV"])
    # the pairs 1e-3 apart have gradients up to 1e6, and positions near 11
    # round by 1.8e-15 in the two frames, 2e-12 of that distance: three such
    # charges of 8009 add 2e-6 sqrt(3 / 8009) to a mean gradient of 35, 1e-9
    assert m["relV"] < 1e-11 and m["reldV"] < 1e-9, m


@pytest.mark.parametrize("kind,kw", [("Laplace", {}), ("Ralpha", {"alpha": -1.5}),
                                     ("Helmholtz", {"k0_r": 0.5, "k0_i": 0.0}),
                                     ("Helmholtz", {"k0_r": 0.5, "k0_i": 0.1})])
def test_dense_cells_mixed_against_oracle(oracle, kind, kw):
    """Mixed V within 1e-6 of the oracle, the gradients within 1e-5; those of
    the charges 1e-3 apart (up to 1e6 where the others have about 35) on
    their own, within 1e-5 of themselves."""
    print("case dense cells mixed", kind, kw, flush=True)
    cx = kind == "Helmholtz"
    coord, q = _charges(8009, cx)
    h = _setup(kind, "mixed", coord, q, "device", 2, 3, **kw)
    assert "dense cells" in h.Print()
    V = h.calcv(q)
    ok = {"Laplace": lambda: oracle.kernel(oracle.LAPLACE, 6, 4.0),
          "Ralpha": lambda: oracle.kernel(oracle.RALPHA, 6, 4.0, alpha=kw.get("alpha", 0.0)),
          "Helmholtz": lambda: oracle.kernel(oracle.HELMHOLTZ, 6, 4.0,
                                             k0=complex(kw.get("k0_r", 0.0), kw.get("k0_i", 0.0)))}[kind]()
    Vo = oracle.calcv(ok, (96, 96, 96), 6, coord, q)
    close = np.r_[20:23, 30:33]
    far = np.setdiff1d(np.arange(len(q)), close)
    rms = lambda x: np.sqrt(np.mean(np.abs(x) ** 2))
    err = [rms(V[far, 0] - Vo[far, 0]) / rms(Vo[far, 0]), rms(V[far, 1:] - Vo[far, 1:]) / rms(Vo[far, 1:]),
           rms(V[close] - Vo[close]) / rms(Vo[close])]
    print(err)
    assert err[0] < 1e-6 and err[1] < 1e-5 and err[2] < 1e-5, err


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_dense_sparse_dense(prec):
    """ResetCoord from dense cells to sparse ones and back: direct sum, order
    and graph are those of a fresh handle, bit for bit."""
    print("case dense sparse dense", prec, flush=True)
    dense, q = _charges(8009, False)
    sparse = uniform_box(8009, 36.0)[0]
    h = _setup("Laplace", prec, dense, q, "device", 2, 3)
    for coord, name in ((dense, "dense cells"), (sparse, "cell rows"), (dense, "dense cells")):
        assert h.ResetCoord(len(q), coord)
        fresh = _setup("Laplace", prec, coord, q, "device", 2, 3)
        assert name in h.Print() and name in fresh.Print()
        V = fresh.calcv(q)
        for _ in range(3):  # launched, captured, replayed
            assert np.array_equal(h.calcv(q), V)
