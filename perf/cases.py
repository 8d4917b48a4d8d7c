"""Performance cases of the CalcV path: what is timed, on which inputs, and how close another correct implementation comes.

A case is one charge set of one kernel and one way of calling the library:

  call "device"  CalcV with the charges and V resident in HBM (npme_calcv_device), one geometry, many charge vectors
  call "host"    the drop-in CalcV on host arrays (copies in and out included)
  call "steps"   two configurations of a trajectory, each ResetCoord + CalcV on host arrays: what a simulation step or a
                 served request costs, set-up included (the two bounding boxes differ, so neither step finds the
                 kernel grid of the other)

Sizes are those of the repository's configurations, tests and benchmark: the request stream (500 to 1M charges at density
0.1, Rdir 8, tol 1e-4 or 1e-6), the 40^3, 100 x 100 x 400, 120^3 and blob configurations, the 50 x 75 x 100 test box.
"""
import functools
import math

import numpy as np
import torch

import npme_amd as N
from npme_amd.inputs import splitmix_uniform, uniform_box

BLOBS, BLOB_SIGMA, BLOB_BOX = 64, 5.0, 400.0


def _case(name, kind, n, box, call="device", precision="mixed", tol=1e-6, Rdir=8.0, Bn=6, alpha=0.0, k0=0.0, k0i=0.0):
    lx, ly, lz = box
    return {"name": name, "kind": kind, "n": n, "lx": lx, "ly": ly, "lz": lz, "call": call, "precision": precision,
            "tol": tol, "Rdir": Rdir, "Bn": Bn, "alpha": alpha, "k0": k0, "k0i": k0i}


def _cube(n, density=0.1):
    return ((n / density) ** (1.0 / 3.0),) * 3


def listed():
    return [
        # the smallest requests of the stream: launches and copies are everything
        _case("laplace_1k_host", "laplace", 1000, _cube(1000), call="host", tol=1e-4),
        # the 40^3 configuration, in FP64 as it is stated
        _case("laplace_10k_fp64", "laplace", 10000, (40.0, 40.0, 40.0), precision="fp64"),
        # a charge count that fills no tile, in the command-line tools' test box, called as the tools call it
        _case("laplace_100k_host", "laplace", 100003, (50.0, 75.0, 100.0), call="host", Rdir=4.0),
        # the benchmark: 1/r at N = 1M, mixed and FP64
        _case("laplace_1m", "laplace", 1000000, _cube(1000000)),
        _case("laplace_1m_fp64", "laplace", 1000000, _cube(1000000), precision="fp64"),
        # r^0.5 in an elongated box
        _case("ralpha_200k", "ralpha", 200000, (100.0, 100.0, 400.0), alpha=0.5),
        # complex charges and grid, wide cutoff
        _case("helmholtz_500k", "helmholtz", 500000, (120.0, 120.0, 120.0), Rdir=10.0, Bn=8, k0=0.5),
        # uneven occupancy: thousands of charges per cell, too many pairs for a list
        _case("blobs_4m", "blobs", 4000000, (BLOB_BOX,) * 3),
        # the erfc split of the 1/r kernel, with the reference's pair set
        _case("erfc_100k", "erfc", 100000, _cube(100000), Rdir=6.0),
        # trajectory steps and served requests: the median request, a large one, a complex one
        _case("steps_laplace_22k", "laplace", 22361, _cube(22361), call="steps", tol=1e-4),
        _case("steps_laplace_600k", "laplace", 600001, _cube(600001), call="steps"),
        _case("steps_helmholtz_50k", "helmholtz", 50000, _cube(50000), call="steps", Bn=8, k0=0.3),
    ]


def draw(rng):
    """One more case of the same ranges: every kernel, call, precision and tolerance above over its sizes."""
    kind = rng.choice(["laplace"] * 5 + ["ralpha"] * 2 + ["helmholtz"] * 2 + ["erfc", "blobs"])
    precision = rng.choice(["mixed", "mixed", "fp64"])
    tol = rng.choice([1e-4, 1e-6])
    top = {"laplace": 1.0e6, "ralpha": 5.0e5, "helmholtz": 3.0e5, "erfc": 1.5e5, "blobs": 4.0e6}[kind]
    low = {"blobs": 2.0e5}.get(kind, 500.0)
    call = rng.choice(["device", "device", "host", "steps"])
    if kind == "blobs":
        call, precision = "device", "mixed"
    n = int(round(math.exp(rng.uniform(math.log(low), math.log(top)))))
    Rdir = rng.choice([6.0, 8.0, 8.0, 10.0]) if kind != "blobs" else 8.0
    Bn = 8 if kind == "helmholtz" else rng.choice([6, 8]) if kind == "laplace" else 6
    alpha = rng.choice([0.5, 1.5]) if kind == "ralpha" else 0.0
    k0 = rng.choice([0.3, 0.5]) if kind == "helmholtz" else 0.0
    if kind == "blobs":
        box = (BLOB_BOX,) * 3
    else:
        # a cube, or a box stretched along one axis
        s = rng.choice([1.0, 1.0, 1.5, 3.0])
        a = (n / (rng.uniform(0.08, 0.2) * s)) ** (1.0 / 3.0)
        box = tuple(rng.sample([a, a, a * s], 3))
    return {k: v for k, v in _case("", kind, n, box, call, precision, tol, Rdir, Bn, alpha, k0).items() if k != "name"}


# ---------------------------------------------------------------- inputs
def _complex(case):
    return case["kind"] == "helmholtz"


def _geometries(case):
    return 2 if case["call"] == "steps" else 1


def _coords(case, seed, step):
    n, box = case["n"], np.array([case["lx"], case["ly"], case["lz"]])
    s = 7919 * int(seed) + 104729 * step
    if case["kind"] != "blobs":
        # a later step's charges fill a slightly larger box
        return splitmix_uniform(s + 1, 3 * n).reshape(n, 3) * (box * (1.0 + 0.002 * step))
    rng = np.random.default_rng(s + 3)
    centre = rng.uniform(0.0, 1.0, (BLOBS, 3)) * box
    return centre[np.arange(n) % BLOBS] + BLOB_SIGMA * rng.standard_normal((n, 3))


def _charges(case, seed):
    n = case["n"]
    if _complex(case):
        rng = np.random.default_rng(7919 * int(seed) + 5)
        return rng.standard_normal(n) + 1j * rng.standard_normal(n)
    q = splitmix_uniform(7919 * int(seed) + 2, n) * 2.0 - 1.0
    return q - q.mean()


def _keywords(case, coord, q):
    func = {"laplace": "Laplace", "blobs": "Laplace", "erfc": "Laplace", "ralpha": "Ralpha", "helmholtz": "Helmholtz"}[case["kind"]]

    def fresh(**kw):
        return N.NPME_KeywordInput(calcType="pme", funcType=func, BnOrder=case["Bn"], Rdir=case["Rdir"], tol=case["tol"],
                                   precision=case["precision"], **kw)

    def fill(k):
        charge = {"chargeComplex": q} if _complex(case) else {"chargeReal": q}
        if not N.NPME_AddMissingKeywords(k, len(q), coord, **charge):
            raise RuntimeError(N.npme_last_error())
        return k

    if case["kind"] == "ralpha":
        # the error model has no row of these exponents: the grid of r^1 serves them
        grid = fill(fresh(alpha=1.0))
        return fill(fresh(alpha=case["alpha"], **{key: grid.GetValue(key) for key in ("N1", "N2", "N3", "n1", "n2", "n3", "nDeriv")}))
    if case["kind"] == "helmholtz":
        return fill(fresh(k0_r=case["k0"], k0_i=case["k0i"]))
    return fill(fresh(EwaldSplit="LaplaceOrig" if case["kind"] == "erfc" else "DerivMatch"))


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.call, s.n = case["call"], case["n"]
    s.coords = [_coords(case, seed, k) for k in range(_geometries(case))]
    s.q = _charges(case, seed)
    keywords = _keywords(case, s.coords[0], s.q)
    set_up = N.NPME_Interface_SetUpComplexKernel if _complex(case) else N.NPME_Interface_SetUpRealKernel
    s.handle = set_up(keywords, s.n, s.coords[0])
    if s.handle is None:
        raise RuntimeError(N.npme_last_error())
    dtype = np.complex128 if _complex(case) else np.float64
    if s.call == "device":
        s.dq = torch.from_numpy(s.q).cuda()
        s.dV = torch.zeros((s.n, 4), dtype=torch.complex128 if _complex(case) else torch.float64, device="cuda")
        torch.cuda.synchronize()
    else:
        s.V = [np.zeros((s.n, 4), dtype) for _ in s.coords]
    return s


def run(s):
    h = s.handle
    if s.call == "device":
        h.calcv_device(s.dV.data_ptr(), s.dq.data_ptr())
        return s.dV
    for coord, V in zip(s.coords, s.V):
        if s.call == "steps" and not h.ResetCoord(s.n, coord):
            raise RuntimeError(N.npme_last_error())
        if not h.CalcV(V, s.n, s.q, coord):
            raise RuntimeError(N.npme_last_error())
    return s.V


# ---------------------------------------------------------------- what a pass cannot do without
@functools.lru_cache(maxsize=None)
def _grid_of(items):
    case = dict(items)
    coord, q = _coords(case, 1, 0), _charges(case, 1)
    k = _keywords(case, coord, q)
    return tuple(int(k.GetValue("N%d" % d)) for d in (1, 2, 3)), int(k.GetValue("nDeriv") or 0)


def _pairs(case):
    """Ordered pairs inside the cutoff, from the charge density."""
    n, R = case["n"], case["Rdir"]
    if case["kind"] == "blobs":
        # the distance of two charges of one blob is Maxwell distributed with scale sqrt(2) sigma
        x = R / (math.sqrt(2.0) * BLOB_SIGMA)
        inside = math.erf(x / math.sqrt(2.0)) - math.sqrt(2.0 / math.pi) * x * math.exp(-0.5 * x * x)
        return n * (n / BLOBS) * inside
    density = n / (case["lx"] * case["ly"] * case["lz"])
    return n * min(n - 1.0, density * 4.0 / 3.0 * math.pi * R ** 3)


def work(case):
    """Per CalcV: positions, charges and the kernel grid read once, V written once; the in-cutoff pairs, one forward and
    one backward transform of the grid, and the spline products of spreading and interpolation."""
    n, cx = case["n"], 2 if _complex(case) else 1
    real = 8 if case["precision"] == "fp64" else 4
    (N1, N2, N3), nder = _grid_of(tuple(sorted((k, v) for k, v in case.items() if k != "name")))
    total = N1 * N2 * N3
    grid = (N1 // 2 + 1) * (N2 // 2 + 1) * (N3 // 2 + 1)
    nbytes = 3 * real * n + 8 * cx * n + 32 * cx * n + real * cx * grid
    flops = _pairs(case) * (20 + 4 * nder) * cx + 2 * 2.5 * cx * total * math.log2(total) + 10 * cx * n * case["Bn"] ** 3
    if case["call"] == "steps":
        nbytes += 24 * n
    return {"bytes": nbytes * _geometries(case), "flops": flops * _geometries(case)}


def tolerance(case):
    """About four times the spread of correct results at the case's precision.  FP64: the neighbour list against the cell
    rows (another order of the pair sums) differs by 2.4e-16 (largest 2.7e-13 of the root mean square), the oracle, whose
    transforms and sums all run in another order, by 1e-14.  Mixed: the two orders differ by up to 2.1e-7 (largest 6e-5),
    FP32 against FP64 by up to 3.8e-7 (largest 8e-5)."""
    if case["precision"] == "fp64":
        return {"rel": 4e-14, "max": 2e-12}
    return {"rel": 1.5e-6, "max": 4e-4}


# ---------------------------------------------------------------- the exact sum
# pairs that the exact sum takes in less than 20 seconds
_MAX_EXACT = {"laplace": 1.1e11, "erfc": 1.1e11, "ralpha": 1.1e11, "helmholtz": 1.1e10, "blobs": 0}


def exact(case, seed):
    """V_t = sum_{s != t} q_s f(r), and its gradient, in FP64 by plain torch."""
    n = case["n"]
    if float(n) * n * _geometries(case) > _MAX_EXACT[case["kind"]]:
        return None
    q = torch.from_numpy(_charges(case, seed)).cuda()
    out = []
    for step in range(_geometries(case)):
        x = torch.from_numpy(_coords(case, seed, step)).cuda()
        V = torch.cat([_exact_rows(case, x, q, t, min(t + _rows(n), n)) for t in range(0, n, _rows(n))])
        out.append(V if case["call"] == "device" else V.cpu().numpy())
    return out[0] if case["call"] == "device" else out


def _rows(n):
    return max(1, min(n, int(2.0e8 / n)))


def _exact_rows(case, x, q, beg, end):
    r = torch.zeros((end - beg, len(x)), dtype=torch.float64, device=x.device)
    for d in range(3):
        r.add_((x[beg:end, d, None] - x[:, d]).square_())
    r.sqrt_()
    own = torch.arange(beg, end, device=x.device)
    row = own - beg
    r[row, own] = 1.0
    parts = [q] if not q.is_complex() else [q.real.contiguous(), q.imag.contiguous()]
    # gradient of f(r): (f'/r)(x_t - x_s), so the sums of f'/r q_s and f'/r q_s x_s suffice
    rhs = torch.stack([c for p in parts for c in (p, p * x[:, 0], p * x[:, 1], p * x[:, 2])], 1)

    def sums(m, columns):
        m[row, own] = 0.0
        return m @ columns

    def gradient(s, t):
        return t * s[:, :1] - s[:, 1:]

    t = x[beg:end]
    if case["kind"] != "helmholtz":
        alpha = case["alpha"] if case["kind"] == "ralpha" else -1.0
        f = r.reciprocal() if alpha == -1.0 else r.pow(alpha)
        g = f.div(r.square_()).mul_(alpha)
        return torch.cat([sums(f, rhs[:, :1]), gradient(sums(g, rhs), t)], 1)
    ri = r.reciprocal()
    damp = ri if case["k0i"] == 0 else ri * torch.exp(-case["k0i"] * r)
    phase = r.mul_(case["k0"])
    c, s = torch.cos(phase).mul_(damp), torch.sin(phase).mul_(damp)
    del phase, r
    # f = c + i s, f'/r = (i k0 - k0i - 1/r) f / r
    a = ri + case["k0i"]
    gr = (-(a * c) - case["k0"] * s).mul_(ri)
    gi = (case["k0"] * c - a * s).mul_(ri)
    vr, vi = sums(c, rhs[:, ::4].contiguous()), sums(s, rhs[:, ::4].contiguous())
    dr, di = sums(gr, rhs), sums(gi, rhs)
    V = torch.complex(vr[:, :1] - vi[:, 1:], vr[:, 1:] + vi[:, :1])
    G = torch.complex(gradient(dr[:, :4], t) - gradient(di[:, 4:], t), gradient(dr[:, 4:], t) + gradient(di[:, :4], t))
    return torch.cat([V, G], 1)
