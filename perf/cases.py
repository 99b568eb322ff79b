"""Workloads of the framework as a user's program runs them, for timing and for comparing outputs.

A case names a model (Wannier functions, range of its R-vectors, which matrices it carries), the
k-points (a Grid, k-lists of adaptive refinement, or a path), the quantity, the Fermi levels and
the precision form.  The models are random Wannier models of the recipe of the repository's own
benchmark: Hermitian in (R, m, n), decaying with |R|, on a bcc lattice, with centres anywhere in
the cell.  `listed()` says for each case what it stands for; `draw()` gives others of the same ranges.

prepare() makes what a program holds before it asks for a result (the System_R, the Grid, lists or
path, the calculators), run() makes one call (run() or run_klists()) and returns its result arrays.
"""
from concurrent.futures import ThreadPoolExecutor
import math
import os

import numpy as np
import torch

import wannierberri_amd as wb

AL, BE = (1, 2, 0), (2, 0, 1)
OPT_FACTOR = 1.602176634e-19 ** 2 / (6.62607015e-34 / (2 * math.pi)) / 1e-10

# what each quantity reads: R-space matrices, and complex nw x nw matrices per k (Ham included)
MATRICES = {"ahc": ("Ham", "AA"), "ahc+bcd": ("Ham", "AA"), "orbital": ("Ham", "AA", "BB", "CC"),
            "orbital-internal": ("Ham",), "tetra": ("Ham", "AA"), "optical": ("Ham", "AA"), "bands": ("Ham", "AA")}
CHANNELS = {"ahc": 10, "ahc+bcd": 37, "orbital": 61, "orbital-internal": 13, "tetra": 10, "optical": 7, "bands": 10}
# complex nw^3 products of the traces per k
PRODUCTS = {"ahc": 0, "ahc+bcd": 18, "orbital": 60, "orbital-internal": 30, "tetra": 0, "optical": 0, "bands": 0}


def _case(name, kind, what, nw, rmax, k, precision="fp64", div="1x1x1", nef=101, ef=1.0, flat=False):
    c = {"kind": kind, "what": what, "nw": nw, "rmax": rmax, "k": k, "precision": precision, "div": div, "nef": nef,
         "ef": ef, "flat": flat}
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # the smallest call: the anomalous Hall conductivity on one small list of refinement points
        _case("klist-8pt-nw8", "klist", "ahc", 8, 2, "8"),
        # a two-band layer model on a dense 2-D grid: many K-blocks of almost no work each
        _case("grid-layer-nw2", "grid", "ahc", 2, 1, "50x50x1", div="4x4x1", nef=1001, ef=3.0, flat=True),
        # bands, velocities and Berry curvature along a path, to be plotted
        _case("path-nw18", "path", "bands", 18, 3, "201"),
        # refinement lists of many sizes in one call
        _case("klist-ragged-nw24", "klist", "ahc", 24, 4, "8,31,17,260,1021,93,2048,640,77,1500,12,405", nef=2001, ef=16.0),
        # the same with a larger basis, in the mixed form
        _case("klist-wide-nw48", "klist", "ahc", 48, 4, "1400,333,2100,65", "fp32", nef=2001, ef=22.0),
        # the benchmark's model and quantities (anomalous Hall conductivity, Berry-curvature dipole)
        # on a part of its grid, in both forms
        _case("grid-berry-nw32", "grid", "ahc+bcd", 32, 4, "16x16x16", div="2x2x1", nef=2001, ef=22.0),
        _case("grid-berry-nw32-mixed", "grid", "ahc+bcd", 32, 4, "16x16x16", "fp32", "2x2x1", 2001, 22.0),
        # a first-principles-sized model with every external matrix, odd sub-grid, a narrow Fermi
        # window (a Fermi sea below it): orbital moment and gyrotropic tensor, sea and surface
        _case("grid-orbital-nw18", "grid", "orbital", 18, 3, "11x9x13", div="2x1x1", nef=501),
        # a large basis, internal terms, levels over the whole spectrum
        _case("grid-orbital-nw64-mixed", "grid", "orbital-internal", 64, 2, "7x7x6", "fp32", nef=2001, ef=20.0),
        # the largest basis
        _case("grid-berry-nw128-mixed", "grid", "ahc+bcd", 128, 2, "6x5x5", "fp32", nef=4001, ef=28.0),
        # the tetrahedron method: conductivity and density of states of a metal
        _case("grid-tetra-nw12", "grid", "tetra", 12, 3, "12x12x12", nef=201),
        # interband optical conductivity, a few Fermi levels by a spectrum of frequencies
        _case("grid-optical-nw18", "grid", "optical", 18, 3, "10x10x10", nef=7),
    ]


def _sizes(text):
    return [int(x) for x in text.split("x")]


def _lists(text):
    return [int(x) for x in text.split(",")]


def _nk(case):
    if case["kind"] == "grid":
        return math.prod(_sizes(case["k"])) * math.prod(_sizes(case["div"]))
    return sum(_lists(case["k"]))


def _nR(case):
    return (2 * case["rmax"] + 1) ** (2 if case["flat"] else 3)


def work(case):
    nw, nk, nR, what = case["nw"], _nk(case), _nR(case), case["what"]
    ncomp = 1 + 3 * (len(MATRICES[what]) - 1)
    out = {"ahc": 3, "ahc+bcd": 12, "orbital": 24, "orbital-internal": 24, "tetra": 4, "optical": 18 * 101}.get(what, 0)
    values = case["nef"] * out if what != "bands" else nk * nw * 7
    nch = CHANNELS[what]
    if case["kind"] == "grid":
        r2k = nk * nch * nw ** 2 * 5 * math.log2(max(2, nk))
    else:
        r2k = 8.0 * nk * nch * nw ** 2 * nR
    eig = nk * (9 if what == "tetra" else 1) * (16 / 3 + 8) * nw ** 3
    rot = nk * (nch - 1) * 16.0 * nw ** 3
    traces = nk * (PRODUCTS[what] * 8.0 * nw ** 3 + 72.0 * nw ** 2)
    if what == "optical":
        traces += nk * 36.0 * nw ** 2 * case["nef"] * 101
    return {"bytes": 16.0 * nR * nw ** 2 * ncomp + 8.0 * values + (24.0 * nk if case["kind"] != "grid" else 0),
            "flops": r2k + eig + rot + traces}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above, no more work than the largest listed one."""
    most = max(work(c)["flops"] for c in listed())
    while True:
        prec = rng.choice(["fp64", "fp32"])
        ef = rng.choice([0.5, 1.0, 3.0, 25.0])
        kind = rng.choice(["klist", "klist", "grid", "grid", "grid", "layer", "path", "orbital", "wide", "tetra", "optical"])
        dims = [rng.randint(7, 17) for _ in range(3)]
        small = "x".join(str(min(d, 11)) for d in dims)
        grid = "x".join(map(str, dims))
        div = "x".join(str(rng.randint(1, 2)) for _ in range(3))
        if kind == "klist":
            lists = ",".join(str(_log(rng, 8, 3000)) for _ in range(rng.randint(1, 8)))
            c = _case(None, "klist", "ahc", _log(rng, 4, 48), rng.randint(2, 4), lists, prec, nef=_log(rng, 101, 2001), ef=ef)
        elif kind == "grid":
            c = _case(None, "grid", rng.choice(["ahc", "ahc+bcd"]), _log(rng, 4, 40), rng.randint(2, 3), grid, prec, div,
                      _log(rng, 101, 2001), ef)
        elif kind == "layer":
            c = _case(None, "grid", "ahc", rng.randint(2, 4), rng.randint(1, 3), "%dx%dx1" % (rng.randint(20, 60), rng.randint(20, 60)),
                      "fp64", "%dx%dx1" % (rng.randint(2, 5), rng.randint(2, 5)), _log(rng, 101, 1001), 3.0, True)
        elif kind == "path":
            c = _case(None, "path", "bands", _log(rng, 4, 32), rng.randint(2, 3), str(_log(rng, 60, 600)), prec)
        elif kind == "orbital":
            c = _case(None, "grid", rng.choice(["orbital", "orbital-internal"]), _log(rng, 6, 40), 2,
                      "x".join(str(rng.randint(5, 9)) for _ in range(3)), prec, "1x1x1", _log(rng, 101, 2001), ef)
        elif kind == "wide":
            c = _case(None, "grid", "ahc+bcd", rng.randint(49, 128), 1, "x".join(str(rng.randint(3, 5)) for _ in range(3)), prec,
                      "1x1x1", _log(rng, 101, 4001), ef)
        elif kind == "tetra":
            c = _case(None, "grid", "tetra", _log(rng, 4, 20), rng.randint(2, 3), small, prec, "1x1x1", _log(rng, 51, 301), 1.0)
        else:
            c = _case(None, "grid", "optical", _log(rng, 4, 28), rng.randint(2, 3), small, prec, "1x1x1", rng.randint(1, 11), 1.0)
        if work(c)["flops"] <= most:
            return c


# -- inputs -----------------------------------------------------------------------


def _model(case, seed):
    """(real lattice, R-vectors, centres, {matrix: [nR, nw, nw, ...]}) from the seed."""
    rng = np.random.Generator(np.random.PCG64([int(seed), case["nw"], case["rmax"]]))
    r = np.arange(-case["rmax"], case["rmax"] + 1)
    lattice = 1.5 * np.array([[-1., 1., 1.], [1., -1., 1.], [1., 1., -1.]])
    if case["flat"]:
        lattice = np.array([[2.5, 0., 0.], [1.25, 2.165, 0.], [0., 0., 8.]])
    iR = np.array([[x, y, z] for x in r for y in r for z in ([0] if case["flat"] else r)])
    nR, nw = len(iR), case["nw"]
    zero = nR // 2
    fall = np.exp(-np.linalg.norm(iR @ lattice, axis=1) / 3.0)

    def gauss(shape, std):
        z = rng.standard_normal((nR,) + shape + (2,)).view(np.complex128)[..., 0]
        z *= (std * fall / math.sqrt(2)).reshape((-1,) + (1,) * len(shape))
        return z

    def hermitian(x):   # the R-vectors run from -R to R, so X(-R) is X read backwards
        return 0.5 * (x + x[::-1].swapaxes(1, 2).conj())

    ham = hermitian(gauss((nw, nw), 1.0))
    ham[zero] += np.diag(rng.uniform(-4.0, 4.0, nw))
    mats = {"Ham": ham}
    for key in MATRICES[case["what"]][1:]:
        x = gauss((nw, nw, 3), 0.1)
        if key != "BB":
            x = hermitian(x)
        if key == "AA":
            x[zero, np.arange(nw), np.arange(nw)] = 0.0
        mats[key] = x
    centres = rng.uniform(0.0, 1.0, (nw, 3)) @ lattice
    return lattice, iR, centres, mats, rng


def _points(case, rng):
    """k-lists around refinement centres, or the nodes of a path (reduced coordinates)."""
    if case["kind"] == "path":
        return rng.uniform(0.0, 1.0, (4, 3))
    return [(rng.uniform(0.0, 1.0, 3) + 0.02 * rng.standard_normal((n, 3))) % 1.0 for n in _lists(case["k"])]


def _path_points(case, nodes):
    """The path as a list of points: straight segments between the nodes."""
    t = np.linspace(0.0, 3.0, _lists(case["k"])[0])
    i = np.minimum(t.astype(int), 2)
    return nodes[i] + (t - i)[:, None] * (nodes[i + 1] - nodes[i])


def _levels(case):
    return np.linspace(-case["ef"], case["ef"], case["nef"])


OMEGA = np.linspace(0.0, 5.0, 101)


def _calculators(case):
    st, Ef, what = wb.calculators.static, _levels(case), case["what"]
    if what == "ahc":
        return {"ahc": st.AHC(Efermi=Ef, constant_factor=1.0)}
    if what == "ahc+bcd":
        return {"ahc": st.AHC(Efermi=Ef, constant_factor=1.0), "bcd": st.BerryDipole_FermiSea(Efermi=Ef)}
    if what in ("orbital", "orbital-internal"):
        kw = dict(Efermi=Ef, constant_factor=1.0)
        return {"ahc": st.AHC(**kw), "morb": st.Morb(**kw), "gme_sea": st.GME_orb_FermiSea(**kw),
                "gme_surf": st.GME_orb_FermiSurf(**kw)}
    if what == "tetra":
        return {"ahc": st.AHC(Efermi=Ef, constant_factor=1.0, tetra=True), "dos": st.DOS(Efermi=Ef, tetra=True)}
    if what == "optical":
        return {"opt": wb.calculators.dynamic.OpticalConductivity(Efermi=Ef, omega=OMEGA, kBT=0.025, smr_fixed_width=0.1)}
    tab = wb.calculators.tabulate
    return {"tab": tab.TabulatorAll({"Energy": tab.Energy(), "velocity": tab.Velocity(), "berry": tab.BerryCurvature()},
                                    mode="path")}


def prepare(case, seed):
    lattice, iR, centres, mats, rng = _model(case, seed)
    system = wb.System_R(lattice, iR, centres, mats, periodic=(True, True, not case["flat"]),
                         force_internal_terms_only=case["what"] == "orbital-internal", name="model")
    state = {"system": system, "calculators": _calculators(case), "kind": case["kind"],
             "parameters_K": {"precision": case["precision"]}}
    if case["kind"] == "grid":
        state["grid"] = wb.Grid(system=system, NKFFT=_sizes(case["k"]), NKdiv=_sizes(case["div"]))
    elif case["kind"] == "path":
        state["grid"] = wb.Path(system=system, k_list=_path_points(case, _points(case, rng)))
    else:
        state["lists"] = _points(case, rng)
    return state


def run(state):
    calcs, par = state["calculators"], state["parameters_K"]
    if state["kind"] == "klist":
        res = wb.run_klists(state["system"], state["lists"], calcs, parameters_K=par)
    else:
        res = wb.run(state["system"], state["grid"], calcs, parameters_K=par, save_files=False, verbose=False)
    if "tab" in calcs:
        return {k: r.data for k, r in res.results["tab"].results.items()}
    return {k: r.data for k, r in res.results.items()}


# -- the same in 64 bits, with torch and numpy alone ---------------------------------


class _Bands:
    """Energies and band-basis matrices of a chunk of k-points: X[name][..., k, n, m]."""

    def __init__(self, case, model, k, dev):
        lattice, iR, centres, mats, _ = model
        c = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(dev)  # noqa: E731
        nw = case["nw"]
        ph = 2 * math.pi * (c(k) @ c(iR).double().T)
        ph = torch.polar(torch.ones_like(ph), ph)
        cR = c((iR @ lattice)[:, None, None, :] + centres[None, None] - centres[None, :, None])

        def to_k(x):
            return (ph @ x.reshape(len(iR), -1)).reshape(len(k), nw, nw)

        ham = to_k(c(mats["Ham"]))
        herm = 0.5 * (ham + ham.mH)
        host = herm.cpu().numpy()
        parts = np.array_split(host, min(len(host), 4 * (os.cpu_count() or 1)))
        with ThreadPoolExecutor(min(16, os.cpu_count() or 1)) as ex:
            got = list(ex.map(np.linalg.eigh, parts))
        self.E = c(np.concatenate([g[0] for g in got]))
        U = c(np.concatenate([g[1] for g in got]))
        self.nw, self.nk, self.dev = nw, len(k), dev
        rot = lambda x: U.mH @ x @ U  # noqa: E731
        X = c(mats["Ham"])
        self.V = [rot(to_k(1j * cR[..., a] * X)) for a in range(3)]
        self.deep = case["what"] in ("ahc+bcd", "orbital", "orbital-internal")
        if self.deep:
            self.W = [[rot(to_k(-cR[..., a] * cR[..., b] * X)) for b in range(3)] for a in range(3)]
        self.ext = case["what"] != "orbital-internal"
        for key, n in (("AA", "A"), ("BB", "B"), ("CC", "C")):
            if key not in mats:
                continue
            Y = [c(mats[key][..., a]) for a in range(3)]
            setattr(self, n, [rot(to_k(y)) for y in Y])
            if self.deep:
                setattr(self, n + "d", [[rot(to_k(1j * cR[..., d] * y)) for d in range(3)] for y in Y])
            if key == "AA" and case["what"] != "optical":
                R = [1j * cR[..., AL[a]] * Y[BE[a]] - 1j * cR[..., BE[a]] * Y[AL[a]] for a in range(3)]
                self.O = [rot(to_k(y)) for y in R]
                if self.deep:
                    self.Od = [[rot(to_k(1j * cR[..., d] * y)) for d in range(3)] for y in R]
        gap = self.E[:, :, None] - self.E[:, None, :]
        self.single = bool((self.E[:, 1:] - self.E[:, :-1] > 1.01e-4).all())
        self.M = torch.where(gap.abs() > 1e-7, 1.0 / torch.where(gap == 0, torch.ones_like(gap), gap), torch.zeros_like(gap))
        self.D = [-v * self.M for v in self.V]

    def omega(self, rows, cols, weight=None):
        """Sum over l in cols of Omega's pair terms, per band n in rows, from (n, l) blocks; the
        within-group terms are the caller's.  weight: a factor per l (the energies, for H)."""
        B = None if not self.ext else self.A if weight is None else self.B
        w = 1.0 if weight is None else weight[:, None, cols]
        out = []
        for al, be in zip(AL, BE):
            D = lambda a: self.D[a][:, rows][:, :, cols]  # noqa: E731
            Dl = lambda a: self.D[a][:, cols][:, :, rows].mT  # noqa: E731
            s = -1j * w * D(al) * Dl(be)
            if self.ext:
                Bl = lambda a: B[a][:, cols][:, :, rows].mT  # noqa: E731
                s = s + D(be) * Bl(al) - D(al) * Bl(be)
            out.append(s)
        return out


def _diag(x):
    return torch.diagonal(x, dim1=-2, dim2=-1)


def _berry(b):
    """Berry curvature per band [3][k, n], every band a group of its own."""
    s = [x.sum(2) for x in b.omega(slice(None), slice(None))]
    return [2 * (x + (0.5 * _diag(b.O[c]) if b.ext else 0)).real for c, x in enumerate(s)]


def _derivatives(b, off):
    """D, its derivative from the right and from the left [b][d], and that of A, between groups
    (off[k, n, l]: n and l in different groups)."""
    on = ~off
    Vi = [v * on for v in b.V]
    D = [-v * b.M * off for v in b.V]
    Mo = b.M * off
    X1, X2, Y1 = [[None] * 3 for _ in range(3)], [[None] * 3 for _ in range(3)], [[None] * 3 for _ in range(3)]
    for p in range(3):
        for d in range(3):
            if d >= p:
                X1[p][d] = X1[d][p] = -Mo * (b.W[p][d] + b.V[p] @ D[d] + b.V[d] @ D[p] - D[p] @ Vi[d] - D[d] @ Vi[p])
                X2[p][d] = X2[d][p] = -Mo * (b.W[p][d] + Vi[p] @ D[d] + Vi[d] @ D[p] - D[p] @ b.V[d] - D[d] @ b.V[p])
            if b.ext:
                Ai = b.A[p] * on
                Y1[p][d] = b.Ad[p][d] - D[d] @ Ai + b.A[p] @ D[d]
    return D, X1, X2, Y1


def _dot(x, y):
    """Diagonal of x y."""
    return (x * y.mT).sum(-1)


def _der_omega(b, off):
    """[c][d] -> per-band DerOmega [k, n] of the partition (off[k, n, l]: l in another group)."""
    D, X1, X2, Y1 = _derivatives(b, off)
    out = [[None] * 3 for _ in range(3)]
    for c in range(3):
        for d in range(3):
            s = 0
            if b.ext:
                s = 0.5 * (_diag(b.Od[c][d]) - _dot(D[d], b.O[c]) + _dot(b.O[c], D[d]))
            for sg, a, e in ((1, AL[c], BE[c]), (-1, BE[c], AL[c])):
                s = s - 1j * sg * _dot(D[a], X1[e][d])
                if b.ext:
                    on = ~off
                    dA = b.Ad[e][d] - D[d] @ (b.A[e] * off) + (b.A[e] * off) @ D[d]
                    s = s - sg * _dot(D[a], Y1[e][d]) - sg * _dot(X2[a][d], b.A[e] * off) \
                        - 1j * sg * _dot(b.A[a] * on, dA)
            out[c][d] = 2 * s.real
    return out


def _der_morb(b, cut):
    """[c][d] -> trace [k] of DerMorb (sign +1) over the bands below the cut."""
    n = torch.arange(b.nw, device=b.dev)
    inn = n < cut
    off = inn[:, None] != inn[None, :]
    off = off[None].expand(b.nk, -1, -1)
    D, X1, X2, Y1 = _derivatives(b, off)
    on = ~off
    E = b.E
    ino = inn.double()
    dom = _der_omega(b, off)
    out = [[None] * 3 for _ in range(3)]
    Ai = [x * on for x in b.A] if b.ext else None
    om = []
    for c in range(3):
        s = -1j * D[AL[c]] @ D[BE[c]]
        if b.ext:
            s = s + 0.5 * b.O[c] - D[AL[c]] @ (b.A[BE[c]] * off) + D[BE[c]] @ (b.A[AL[c]] * off) - 1j * Ai[AL[c]] @ Ai[BE[c]]
        om.append(s + s.mH)
    for c in range(3):
        for d in range(3):
            Vi = b.V[d] * on
            s = -2j * _dot(D[AL[c]] @ Vi, D[BE[c]])
            if b.ext:
                s = s + _diag(b.Cd[c][d]) - _dot(D[d], b.C[c] * off) + _dot(b.C[c] * off, D[d]) - 2j * _dot(Ai[AL[c]] @ Vi, Ai[BE[c]])
            for sg, a, e in ((1, AL[c], BE[c]), (-1, BE[c], AL[c])):
                s = s - 2j * sg * _dot(D[a] * E[:, None, :], X1[e][d])
                if b.ext:
                    dA = b.Ad[e][d] - D[d] @ (b.A[e] * off) + (b.A[e] * off) @ D[d]
                    dB = b.Bd[e][d] - D[d] @ (b.B[e] * on) + (b.B[e] * on) @ D[d]
                    s = s - 2j * sg * _dot(Ai[a] * E[:, None, :], dA) - 2 * sg * _dot(D[a], dB) \
                        - 2 * sg * ((b.B[a] * off).conj() * X1[e][d]).sum(-2)
            v = s.real + E * dom[c][d] + _dot(om[c] * on, Vi).real
            out[c][d] = (v * ino).sum(-1)
    return out


def _scan(case, E, values, fder):
    """Sums over k and bands at every Fermi level: values [k, n, ...] -> [nEF, ...]."""
    Ef = _levels(case)
    dE = Ef[1] - Ef[0]
    extra = 1 if fder else 0
    lo, n = Ef[0] - extra * dE, len(Ef) + 2 * extra
    at = torch.ceil((E - lo) / dE).long().clamp(min=0)
    use = E <= Ef[-1] + extra * dE
    if fder:
        use = use & (E >= lo)
    at = torch.where(use & (at < n), at, torch.full_like(at, n)).reshape(-1)
    flat = values.reshape(at.shape[0], -1)
    hist = torch.zeros((n + 1, flat.shape[1]), dtype=torch.float64, device=E.device)
    hist.index_add_(0, at, flat)
    hist = hist[:n].cumsum(0)
    if fder:
        hist = (hist[2:] - hist[:-2]) / (2 * dE)
    return hist.reshape((len(Ef),) + values.shape[2:])


def _grid_points(case):
    N, div = _sizes(case["k"]), _sizes(case["div"])
    g = np.stack(np.meshgrid(*[np.arange(n) for n in N], indexing="ij"), -1).reshape(-1, 1, 3)
    s = np.stack(np.meshgrid(*[np.arange(n) for n in div], indexing="ij"), -1).reshape(1, -1, 3)
    return ((g + s / np.array(div)) / np.array(N)).reshape(-1, 3)


def _tetra_weight(Ef, e):
    """Occupied fraction of tetrahedra with corner energies e [..., 4] at Ef [n] -> [..., n], and its slope."""
    e = torch.sort(e, -1).values
    split = torch.tensor([0.0, 1.0, 2.0, 3.0], device=e.device, dtype=e.dtype) * 1e-12
    e1, e2, e3, e4 = (x[..., None] for x in (e + split).unbind(-1))
    x = Ef
    u, v = x - e1, x - e4
    lo = u ** 3 / ((e2 - e1) * (e3 - e1) * (e4 - e1))
    hi = 1 + v ** 3 / ((e4 - e1) * (e4 - e2) * (e4 - e3))
    a13, a14, a23, a24 = u / (e3 - e1), u / (e4 - e1), (x - e2) / (e3 - e2), (x - e2) / (e4 - e2)
    mid = a23 * a24 + a13 * (a14 * (1 - a24) + a24 * (1 - a23))
    occ = torch.where(x < e1, 0.0, torch.where(x < e2, lo, torch.where(x < e3, mid, torch.where(x < e4, hi, 1.0))))
    d13, d14, d23, d24 = 1 / (e3 - e1), 1 / (e4 - e1), 1 / (e3 - e2), 1 / (e4 - e2)
    slope_mid = d23 * a24 + a23 * d24 + d13 * (a14 * (1 - a24) + a24 * (1 - a23)) \
        + a13 * (d14 * (1 - a24) - a14 * d24 + d24 * (1 - a23) - a24 * d23)
    slope = torch.where(x < e1, 0.0, torch.where(x < e2, 3 * lo / u, torch.where(x < e3, slope_mid, torch.where(
        x < e4, 3 * (hi - 1) / v, 0.0))))
    return occ, slope


def _tetra(case, model, b, k, dev):
    """AHC and DOS of the tetrahedron method for a chunk of k."""
    half = 0.5 / (np.array(_sizes(case["k"])) * np.array(_sizes(case["div"])))
    corner = {}
    for i in range(8):
        sh = np.array([i >> 2 & 1, i >> 1 & 1, i & 1])
        lattice, iR, centres, mats, _ = model
        ph = 2 * math.pi * torch.from_numpy((k + (2 * sh - 1) * half) @ iR.T).to(dev)
        ham = (torch.polar(torch.ones_like(ph), ph) @ torch.from_numpy(mats["Ham"].reshape(len(iR), -1)).to(dev))
        ham = ham.reshape(len(k), b.nw, b.nw)
        corner[tuple(sh)] = torch.from_numpy(np.linalg.eigvalsh((0.5 * (ham + ham.mH)).cpu().numpy())).to(dev)
    tets = []
    for side in (0, 1):
        for axis in range(3):
            f = lambda p, q: corner[tuple(np.insert([p, q], axis, side))]  # noqa: E731, B023
            tets += [(f(0, 0), f(0, 1), f(1, 1)), (f(0, 0), f(1, 0), f(1, 1))]
    Ef = torch.from_numpy(_levels(case)).to(dev)
    occ = slope = 0
    for t in tets:
        o, s = _tetra_weight(Ef, torch.stack((b.E,) + t, -1))
        occ, slope = occ + o / 12, slope + s / 12
    om = torch.stack(_berry(b), -1)
    return {"ahc": torch.einsum("kne,knc->ec", occ, om), "dos": slope.sum((0, 1))}


def _orbital(case, b):
    out = {}
    om = torch.stack(_berry(b), -1)
    nw, E = b.nw, b.E
    Ef = torch.from_numpy(_levels(case)).to(b.dev)
    out["ahc"] = ahc = _scan(case, E, om, 0)
    pair = b.omega(slice(None), slice(None))
    hpair = b.omega(slice(None), slice(None), weight=E)
    # orbital moment of one band, for the surface term
    hb = [2 * (h.sum(2) + (0.5 * _diag(b.C[c]) if b.ext else 0)).real + E * om[..., c] for c, h in enumerate(hpair)]
    v = torch.stack([_diag(x).real for x in b.V], -1)
    surf = _scan(case, E, v[..., :, None] * torch.stack(hb, -1)[..., None, :], 1)
    dip = _scan(case, E, v[..., :, None] * om[..., None, :], 1)
    out["gme_surf"] = surf - 2 * Ef[:, None, None] * dip
    # sums over the bands below each cut
    morb = torch.zeros((b.nk, nw + 1, 3), dtype=torch.float64, device=b.dev)
    der = torch.zeros((b.nk, nw + 1, 3, 3), dtype=torch.float64, device=b.dev)
    dom_all = _der_omega(b, ~torch.eye(nw, dtype=torch.bool, device=b.dev)[None].expand(b.nk, -1, -1))
    for cut in range(1, nw + 1):
        i, o = slice(0, cut), slice(cut, nw)
        for c in range(3):
            s = (hpair[c] + E[:, :, None] * pair[c])[:, i, o].sum((1, 2))
            if b.ext:
                aa = b.A[AL[c]][:, i, i] * b.A[BE[c]][:, i, i].mT
                s = s + (0.5 * _diag(b.C[c]) + 0.5 * E * _diag(b.O[c]))[:, i].sum(1) \
                    - 1j * (aa * (E[:, None, i] + E[:, i, None])).sum((1, 2))
            morb[:, cut, c] = 2 * s.real
        dm = _der_morb(b, cut)
        for c in range(3):
            for d in range(3):
                der[:, cut, c, d] = dm[c][d]
    morb = _scan(case, E, morb[:, 1:] - morb[:, :-1], 0)
    out["morb"] = morb - 2 * Ef[:, None] * ahc
    der = _scan(case, E, (der[:, 1:] - der[:, :-1]).transpose(2, 3), 0)
    bcd = _scan(case, E, torch.stack([torch.stack([dom_all[c][d] for c in range(3)], -1) for d in range(3)], -2), 0)
    out["gme_sea"] = der - 2 * Ef[:, None, None] * bcd
    return out


def _optical(case, b):
    Ef, om = torch.from_numpy(_levels(case)).to(b.dev), torch.from_numpy(OMEGA).to(b.dev)
    A = [1j * d + a for d, a in zip(b.D, b.A)]
    M = torch.stack([torch.stack([1j * A[p] * A[q].mT for q in range(3)], -1) for p in range(3)], -2).reshape(b.nk, -1, 9)
    f = 1 / (torch.exp(((b.E[..., None] - Ef) / 0.025).clamp(-700, 700)) + 1)
    f = torch.where(Ef > b.E[..., None] + 30 * 0.025, 1.0, torch.where(Ef < b.E[..., None] - 30 * 0.025, 0.0, f))
    fE = (f[:, None] - f[:, :, None]).reshape(b.nk, -1, len(Ef))
    de = (b.E[:, None] - b.E[:, :, None]).reshape(b.nk, -1)
    out = 0
    for k in range(b.nk):
        fw = de[k][:, None] / (de[k][:, None] - om - 0.1j)
        out = out + torch.einsum("pe,pw,px->ewx", fE[k].to(M.dtype), fw, M[k])
    return {"opt": out.reshape(len(Ef), len(om), 3, 3)}


def exact(case, seed):
    if case["what"].startswith("orbital") and _nk(case) * case["nw"] ** 4 > 6e9:
        return None   # a product per band cut: longer than the other cases together
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    model = _model(case, seed)
    lattice, what = model[0], case["what"]
    if case["kind"] == "grid":
        k = _grid_points(case)
    else:
        pts = _points(case, model[4])
        k = _path_points(case, pts) if case["kind"] == "path" else np.concatenate(pts)
    step = max(1, int(4e8 / (16 * CHANNELS[what] * case["nw"] ** 2 * (4 if what.startswith("orb") or "bcd" in what else 2))))
    if what in ("tetra", "optical"):
        step = min(step, 64)
    total, rows = {}, []
    for k0 in range(0, len(k), step):
        b = _Bands(case, model, k[k0:k0 + step], dev)
        if not b.single:
            return None   # degenerate bands form groups
        if what == "bands":
            rows.append((b.E, torch.stack([_diag(x).real for x in b.V], -1), torch.stack(_berry(b), -1)))
            continue
        if what == "tetra":
            part = _tetra(case, model, b, k[k0:k0 + step], dev)
        elif what == "optical":
            part = _optical(case, b)
        elif what.startswith("orbital"):
            part = _orbital(case, b)
        else:
            part = {"ahc": _scan(case, b.E, torch.stack(_berry(b), -1), 0)}
            if what == "ahc+bcd":
                der = _der_omega(b, ~torch.eye(b.nw, dtype=torch.bool, device=dev)[None].expand(b.nk, -1, -1))
                part["bcd"] = _scan(case, b.E, torch.stack([torch.stack([der[c][d] for c in range(3)], -1)
                                                            for d in range(3)], -2), 0)
        total = {q: total[q] + v if q in total else v for q, v in part.items()}
    if what == "bands":
        e, v, o = (torch.cat(x).cpu().numpy() for x in zip(*rows))
        return {"Energy": e, "velocity": v, "berry": o}
    volume = abs(np.linalg.det(lattice))
    scale = {q: 1.0 / len(k) / volume for q in total}
    for q in ("morb", "dos"):
        if q in scale:
            scale[q] *= volume
    if "opt" in scale:
        scale["opt"] *= OPT_FACTOR
    return {q: (v * scale[q]).cpu().numpy() for q, v in total.items()}
