"""Edges of the kernels' tiles and dispatch rules: the smallest and largest sizes of each variant,
remainders, and inputs whose route differs.  Tolerances follow from the arithmetic (unit roundoff
times the length of the sums times the norms), with a factor for the worst case over the samples."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.fixture(scope="module")
def ctx():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from wannierberri_amd import _lib
    return _lib.get_context(0)


def _hermitian(rng, nk, nw):
    H = rng.standard_normal((nk, nw, nw)) + 1j * rng.standard_normal((nk, nw, nw))
    return 0.5 * (H + H.conj().swapaxes(1, 2)) + np.diag(np.linspace(-4, 4, nw))


@pytest.mark.parametrize("nw", [1, 2, 3, 4, 7, 10, 15, 22, 33, 34, 50, 62, 66, 67, 126, 128])
def test_eigh_sizes(ctx, nw):
    """One size of each kind of the FP32 Jacobi kernels (one wave, four waves, V in registers; odd
    sizes have a padding index): residual, orthogonality and order against the input."""
    import torch
    from wannierberri_amd import _lib
    nk = 5
    H = _hermitian(np.random.default_rng(nw), nk, nw)
    Hd = torch.from_numpy(H).cuda()
    norm = np.linalg.norm(H, 2, axis=(1, 2)).max()
    Eref = np.linalg.eigvalsh(H)
    for prec, cd, eps in ((_lib.WBMI_F64, torch.complex128, EPS), (_lib.WBMI_F32, torch.complex64, 6e-8)):
        E = torch.empty((nk, nw), dtype=torch.float64, device="cuda")
        U = torch.empty((nk, nw, nw), dtype=cd, device="cuda")
        if prec == _lib.WBMI_F64:
            ctx.eigh(Hd, nw * nw, E, U, prec, nw, refine=16)
        else:
            ctx.eigh(None, nw * nw, E, U, prec, nw, refine=16, H64=Hd)
        E, U = E.cpu().numpy(), U.cpu().numpy().astype(complex)
        assert np.all(np.diff(E, axis=1) >= 0)
        assert np.abs(E - Eref).max() < 8 * EPS * nw * norm
        assert np.abs(H @ U - U * E[:, None, :]).max() < 8 * eps * nw * norm
        assert np.abs(U.conj().swapaxes(1, 2) @ U - np.eye(nw)).max() < 8 * eps * nw


@pytest.mark.parametrize("nw", [5, 16, 17, 32, 44, 45, 48, 49, 64, 65])
@pytest.mark.parametrize("gap", [1.0, 1e-9])
def test_eigh_refine_blocks(ctx, nw, gap):
    """The refinement at the edges of its 16 x 16 blocks, without and with a pair of eigenvalues so close
    that the correction steps leave it mixed (the Jacobi pass over clusters)."""
    import torch
    from wannierberri_amd import _lib
    rng = np.random.default_rng(nw)
    nk = 3
    E = np.cumsum(0.5 + rng.random((nk, nw)), axis=1)
    E[:, nw // 2] = E[:, nw // 2 - 1] + gap * (0.5 if gap == 1.0 else 1.0)
    V = np.linalg.qr(rng.standard_normal((nk, nw, nw)) + 1j * rng.standard_normal((nk, nw, nw)))[0]
    H = (V * E[:, None, :]) @ V.conj().swapaxes(1, 2)
    H = 0.5 * (H + H.conj().swapaxes(1, 2))
    norm = np.abs(E).max()
    Ed = torch.empty((nk, nw), dtype=torch.float64, device="cuda")
    U = torch.empty((nk, nw, nw), dtype=torch.complex128, device="cuda")
    ctx.eigh(torch.from_numpy(H).cuda(), nw * nw, Ed, U, _lib.WBMI_F64, nw, refine=16)
    e, u = Ed.cpu().numpy(), U.cpu().numpy()
    assert np.abs(e - np.linalg.eigvalsh(H)).max() < 8 * EPS * nw * norm
    assert np.abs(H @ u - u * e[:, None, :]).max() < 8 * EPS * nw * norm
    assert np.abs(u.conj().swapaxes(1, 2) @ u - np.eye(nw)).max() < 8 * EPS * nw


@pytest.mark.parametrize("nw", [45, 64])
def test_eigh_needs_no_workspace(ctx, nw):
    """Refined solves of up to 64 bands without a workspace: more k-points than the no-allocation form's scratch
    would hold at four matrices each."""
    import torch
    from wannierberri_amd import _lib
    nk = _lib.lib().wbmi_eigh_noalloc_max_bytes() // (4 * 16 * nw * nw) + 3
    H = torch.from_numpy(_hermitian(np.random.default_rng(nw), 3, nw)).cuda()[torch.arange(nk) % 3].contiguous()
    E = torch.empty((nk, nw), dtype=torch.float64, device="cuda")
    U = torch.empty((nk, nw, nw), dtype=torch.complex128, device="cuda")
    ctx.eigh_noalloc(H, nw * nw, E, U, _lib.WBMI_F64, nw, refine=16)
    assert torch.equal(E, E[torch.arange(nk) % 3])
    assert np.abs(E[:3].cpu().numpy() - np.linalg.eigvalsh(H[:3].cpu().numpy())).max() < 8 * EPS * nw * 20
    L, E1, U1 = _lib.lib(), torch.empty_like(E), torch.empty_like(U)
    assert L.wbmi_eigh(ctx.h, nk, nw, _lib._ptr(H), nw * nw, _lib._ptr(E1), _lib._ptr(U1), _lib.WBMI_F64, 16, None, None, 0) == 0
    assert torch.equal(E, E1) and torch.equal(U, U1)


@pytest.mark.parametrize("nw", [33, 40, 64])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_eigh_repeats(ctx, nw, prec):
    """Energies of 33 to 64 bands are the same bits in every call (their norms are summed by three or four
    waves)."""
    import torch
    from wannierberri_amd import _lib
    p, cd = ((_lib.WBMI_F64, torch.complex128) if prec == "fp64" else (_lib.WBMI_F32, torch.complex64))
    nk = 6000 if nw < 64 else 4000
    H = torch.from_numpy(_hermitian(np.random.default_rng(nw), nk, nw)).cuda()
    first = None
    for _ in range(25):
        E = torch.empty((nk, nw), dtype=torch.float64, device="cuda")
        U = torch.empty((nk, nw, nw), dtype=cd, device="cuda")
        if prec == "fp64":
            ctx.eigh(H, nw * nw, E, U, p, nw, refine=16)
        else:
            ctx.eigh(None, nw * nw, E, U, p, nw, refine=16, H64=H)
        first = E if first is None else first
        assert torch.equal(E, first)


@pytest.mark.parametrize("nw", [16, 17, 32, 33, 50, 64])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_eigh_waves_per_k(ctx, nw, prec):
    """A k-point's eigenvectors and energies do not depend on the number of k-points of the call (few:
    more waves per k-point in the Jacobi kernel, the same operations per element), nor does a warm start."""
    import torch
    from wannierberri_amd import _lib
    p, cd = ((_lib.WBMI_F64, torch.complex128) if prec == "fp64" else (_lib.WBMI_F32, torch.complex64))
    H = torch.from_numpy(_hermitian(np.random.default_rng(nw), 7, nw)).cuda()
    out = []
    for nk in (7, 1001):
        Hn = H[torch.arange(nk) % 7].contiguous()
        E = torch.empty((nk, nw), dtype=torch.float64, device="cuda")
        U = torch.empty((nk, nw, nw), dtype=cd, device="cuda")
        def solve(U0=None):
            if prec == "fp64":
                ctx.eigh(Hn, nw * nw, E, U, p, nw, refine=16, U0=U0)
            else:
                ctx.eigh(None, nw * nw, E, U, p, nw, refine=16, H64=Hn, U0=U0)
        solve()
        U1 = U.clone()
        solve(U0=U1.roll(1, 0).contiguous() if nk == 7 else U1[(torch.arange(nk) + 6) % 7].contiguous())
        out.append((E[:7].clone(), U1[:7], U[:7].clone()))
    for a, b in zip(*out):
        # complex128 sums of norms may be taken in another order (a step's threshold); complex64 is stored
        assert (a - b).abs().max().item() <= (16 * EPS * nw * 10 if a.dtype != torch.complex64 else 0.0)


@pytest.mark.parametrize("nw,ef,precision", [(3, 0.6, "fp64"), (16, 1.0, "fp64"), (17, 1.0, "fp32"), (24, 40.0, "fp64"),
                                             (32, 1.0, "fp64"), (32, 1.0, "fp32"), (33, 1.5, "fp64")])
def test_scan_sea_and_split(ctx, nw, ef, precision):
    """DerOmega, DerMorb, Omega and Morb on a few k-points (several workgroups share each one's tasks)
    with a Fermi sea of many bands below a narrow window, or every band in range: against the oracle,
    on models with two bands 5e-5 apart at every k-point (one group)."""
    import wannierberri_amd as wb
    from oracle import wb_oracle as O
    from wannierberri_amd import models
    s = models.synthetic(num_wann=nw, Rmax=1, seed=50 + nw, with_BBCC=True)
    ham = s.get_R_mat("Ham").copy()
    # the last two orbitals decoupled from the rest and from each other: a pair 5e-5 apart
    ham[:, -2:, :] = 0.
    ham[:, :, -2:] = 0.
    i0 = s.rvec.iR0
    ham[i0, -2, -2], ham[i0, -1, -1] = -3.0, -3.0 + 5e-5
    s.set_R_mat("Ham", ham, reset=True)
    Ef = np.linspace(-ef, ef, 13)
    k = np.random.default_rng(nw).random((3, 3))
    st = wb.calculators.static
    calcs = {"ahc": st.AHC(Efermi=Ef), "bcd": st.BerryDipole_FermiSea(Efermi=Ef), "morb": st.Morb(Efermi=Ef),
             "gme": st.GME_orb_FermiSea(Efermi=Ef)}
    got = wb.run_klists(s, [k], calcs, parameters_K={"precision": precision})
    o = O.OracleSystem(s.real_lattice, s.rvec.iRvec, s.wannier_centers_cart,
                       {m: s.get_R_mat(m) for m in ("Ham", "AA", "BB", "CC")})
    d = O.OracleDataK(o, k_list=k)
    for name, calc in (("ahc", O.AHC(Ef)), ("bcd", O.BerryDipole_FermiSea(Ef)), ("morb", O.Morb(Ef)),
                       ("gme", O.GME_orb_FermiSea(Ef))):
        ref = calc(d).data
        err = np.abs(got.results[name].data - ref).max() / np.abs(ref).max()
        print(f"test_scan_sea_and_split nw={nw} {precision} {name}: {err:.2e}", flush=True)
        # the close pair's denominators are cut out of the sums (one group); the rest is of order one
        assert err < (1e-9 if precision == "fp64" else 2e-5), name


@pytest.mark.parametrize("nw,ef,precision,terms", [
    (2, 40.0, "fp64", "in"), (15, 40.0, "fp64", "in"), (16, 1.0, "fp32", "in"), (17, 40.0, "fp64", "in"),
    (17, 40.0, "fp32", "in"), (33, 40.0, "fp32", "in"), (49, 2.0, "fp64", "in"), (100, 1.0, "fp64", "in"),
    (16, 40.0, "fp64", "ex"), (17, 40.0, "fp64", "ex"), (16, 40.0, "fp64", "both"), (17, 1.0, "fp32", "both"),
    (33, 40.0, "fp64", "both")])
def test_scan_all_cuts(nw, ef, precision, terms):
    """The non-additive formulas (Morb, DerMorb) at the edges of the 16-band blocks, with every border in
    the levels' range or few of them: internal terms, external terms and both, against the oracle."""
    import wannierberri_amd as wb
    from oracle import wb_oracle as O
    from wannierberri_amd import models
    s = models.synthetic(num_wann=nw, Rmax=1, seed=70 + nw, with_BBCC=True)
    Ef = np.linspace(-ef, ef, 9)
    k = np.random.default_rng(nw).random((2, 3))
    st = wb.calculators.static
    kw = dict(kwargs_formula={"internal_terms": terms != "ex", "external_terms": terms != "in"})
    got = wb.run_klists(s, [k], {"morb": st.Morb(Efermi=Ef, **kw), "gme": st.GME_orb_FermiSea(Efermi=Ef, **kw)},
                        parameters_K={"precision": precision})
    o = O.OracleSystem(s.real_lattice, s.rvec.iRvec, s.wannier_centers_cart,
                       {m: s.get_R_mat(m) for m in ("Ham", "AA", "BB", "CC")})
    d = O.OracleDataK(o, k_list=k)
    for name, calc in (("morb", O.Morb(Ef, **kw)), ("gme", O.GME_orb_FermiSea(Ef, **kw))):
        ref = calc(d).data
        err = np.abs(got.results[name].data - ref).max() / np.abs(ref).max()
        print(f"test_scan_all_cuts nw={nw} {precision} {terms} {name}: {err:.2e}", flush=True)
        # sums of 1 / dE^3 over gaps above 1e-4 (the group threshold), typically 1e-2: 1e-16 * 1e6 and a margin
        assert err < (1e-9 if precision == "fp64" else 2e-5), name


@pytest.mark.parametrize("nw,precision,kramers", [
    (2, "fp64", False), (7, "fp64", False), (8, "fp32", True), (9, "fp64", True), (17, "fp32", False), (24, "fp64", True),
    (25, "fp64", False), (33, "fp32", False), (49, "fp64", True), (65, "fp64", False)])
def test_scan_diagonal_traces(nw, precision, kramers):
    """Omega and the velocity products with Omega and Morb_Hpm at the edges of the 8 x 8 blocks, groups of one
    band, a pair 5e-5 apart, or every two bands a group: against the oracle."""
    import wannierberri_amd as wb
    from oracle import wb_oracle as O
    from wannierberri_amd import models
    s = models.synthetic(num_wann=nw, Rmax=1, seed=90 + nw, with_BBCC=True)
    ham = s.get_R_mat("Ham").copy()
    ham[:, -2:, :] = 0.
    ham[:, :, -2:] = 0.
    i0 = s.rvec.iR0
    ham[i0, -2, -2], ham[i0, -1, -1] = 0.5, 0.5 + 5e-5
    s.set_R_mat("Ham", ham, reset=True)
    Ef = np.linspace(-40., 40., 41)
    k = np.random.default_rng(nw).random((3, 3))
    st = wb.calculators.static
    kw = dict(degen_Kramers=kramers)
    names = {"ahc": "AHC", "bcd": "BerryDipole_FermiSurf", "gme": "GME_orb_FermiSurf"}
    got = wb.run_klists(s, [k], {n: getattr(st, c)(Efermi=Ef, **kw) for n, c in names.items()},
                        parameters_K={"precision": precision})
    o = O.OracleSystem(s.real_lattice, s.rvec.iRvec, s.wannier_centers_cart,
                       {m: s.get_R_mat(m) for m in ("Ham", "AA", "BB", "CC")})
    d = O.OracleDataK(o, k_list=k)
    for name, c in names.items():
        ref = getattr(O, c)(Ef, **kw)(d).data
        err, scale = np.abs(got.results[name].data - ref).max(), np.abs(ref).max()   # (zero at nw = 2: flat bands)
        print(f"test_scan_diagonal_traces nw={nw} {precision} {name}: {err:.2e} of {scale:.2e}", flush=True)
        # sums of 1 / dE^2 over gaps above 1e-4 between groups, typically 1e-2: 1e-16 * 1e4 and a margin
        assert err <= (1e-9 if precision == "fp64" else 2e-5) * scale, name


def _off_mirror(nw, external, group=1):
    """Complex64 channels of two k-points with V Hermitian to storage rounding only: one element of the
    matrix before its rotation is off its mirror, so every element after it is, the diagonal among them.  Every
    `group` bands (5e-5 apart) a group in a bin of its own, two groups 4e-3 apart.  Returns the channels (V, W;
    A, A', rotA, rotA'), E, bin width, the bin of each band, and the oracle's K-block on the same stored matrices."""
    from oracle import wb_oracle as O
    rng = np.random.default_rng(nw)
    nk, dEF = 2, 2e-3
    ng = -(-nw // group)
    step = np.full((nk, ng), 125)
    step[:, ng // 2] = 2
    level = np.cumsum(step + (step > 2) * rng.integers(0, 9, (nk, ng)), axis=1)   # the bin of each group
    level = np.repeat(level, group, axis=1)[:, :nw]
    def herm(n):
        x = rng.standard_normal((nk, n, nw, nw)) + 1j * rng.standard_normal((nk, n, nw, nw))
        return (0.5 * (x + x.conj().swapaxes(2, 3))).astype(np.complex64).astype(complex)
    U = np.linalg.qr(rng.standard_normal((nk, nw, nw)) + 1j * rng.standard_normal((nk, nw, nw)))[0]
    V, W = herm(3), herm(9)
    W = 0.5 * (W + W[:, [0, 3, 6, 1, 4, 7, 2, 5, 8]])
    V[:, :, 1, 0] += 6e-8
    X = np.concatenate([V, W], axis=1)
    X = (U.conj().swapaxes(1, 2)[:, None] @ X @ U[:, None]).astype(np.complex64)
    if external:
        X = np.concatenate([X, herm(24).astype(np.complex64)], axis=1)
    E = (level - 0.5) * dEF + 5e-5 * (np.arange(nw) % group)
    x = np.moveaxis(X.astype(complex), 1, 3)
    bar = {("Ham", 1): x[..., :3], ("Ham", 2): x[..., 3:12].reshape(nk, nw, nw, 3, 3)}
    if external:
        bar.update({("AA", 0): x[..., 12:15], ("AA", 1): x[..., 15:24].reshape(nk, nw, nw, 3, 3),
                    ("rotAA", 0): x[..., 24:27], ("rotAA", 1): x[..., 27:].reshape(nk, nw, nw, 3, 3)})

    class Given(O.OracleDataK):
        E_K = E
        force_internal_terms_only = False

        def __init__(self):
            self._cov = {}

        def Xbar(self, name, der=0):
            return bar[name, der]
    return X, E, dEF, level, Given()


def _scan_bins(ctx, X, E, dEF, level, formula, external):
    import torch
    from wannierberri_amd import _lib
    nbin = int(level.max()) + 2
    p = _lib.ScanParams()
    p.formula, p.sign, p.internal_terms, p.external_terms, p.fder = formula, 1, 1, int(external), 0
    p.nEF_extra, p.EFmin, p.EFmax, p.dEF, p.degen_thresh = nbin, 0.0, (nbin - 1) * dEF, dEF, 1e-4
    for i in range(_lib.NROLES):
        p.ch[i] = i if i < X.shape[1] else -1   # V, W, A, A', rotA, rotA' have the first roles in this order
    hist = torch.zeros((nbin, 9), dtype=torch.float64, device="cuda")
    ctx.static_scan(torch.from_numpy(E).cuda(), torch.from_numpy(X).cuda(), _lib.WBMI_F32, p, 1.0, hist)
    return hist.cpu().numpy()


@pytest.mark.parametrize("nw", [7, 16, 32, 33, 70])
def test_scan_velocity_off_its_mirror(ctx, nw):
    """DerOmega and DerMorb (internal terms; with them the gyrotropic tensor and the Berry-curvature dipole)
    against the oracle's formulas on the same stored matrices."""
    from oracle import wb_oracle as O
    from wannierberri_amd import _lib
    X, E, dEF, level, d = _off_mirror(nw, False)
    for formula, f in ((_lib.FORMULA_DEROMEGA, O.DerOmega(d, external_terms=False)),
                       (_lib.FORMULA_DERMORB, O.DerMorb(d, sign=1, external_terms=False))):
        hist = _scan_bins(ctx, X, E, dEF, level, formula, False)
        ref = np.zeros_like(hist)
        for ik in range(len(E)):
            bands = np.arange(nw)
            cuts = np.zeros((nw + 1, 9))
            for c in range(1, nw + 1):
                # tr (Omega V + V Omega) / 2, Omega = s + s^+, is formed as 2 Re tr s V (V read as Hermitian here)
                D, v = d.D_H[ik], d.Xbar("Ham", 1)[ik, :c, :c]
                s = -1j * np.einsum("mlc,lnc->mnc", D[:c, c:][..., [1, 2, 0]], D[c:, :c][..., [2, 0, 1]])
                herm = np.einsum("mnc,nmd->cd", s, v) - np.einsum("nmc,nmd->cd", s.conj(), v)
                cuts[c] = (f.trace(ik, bands[:c], bands[c:]) + herm.real).reshape(9)
            for n in range(nw):
                value = cuts[n + 1] - cuts[n] if formula == _lib.FORMULA_DERMORB else \
                    f.trace(ik, bands[n:n + 1], np.delete(bands, n)).reshape(9)
                ref[level[ik, n]] += value
        err = np.abs(hist - ref).max() / np.abs(ref).max()
        print(f"test_scan_velocity_off_its_mirror nw={nw} formula {formula}: {err:.1e}", flush=True)
        # about 3 nw roundings of terms of the size of the largest (5e-14 at nw = 70); the energies' differences
        # are exact.  A real V_nn is off by 1e-9 .. 1e-8: Im V_nn / (V_nn - V_ll)
        assert err < 1e-12, formula


@pytest.mark.parametrize("nw,group", [(7, 1), (16, 1), (32, 1), (33, 1), (70, 1), (7, 2), (18, 2), (32, 4), (33, 2), (70, 3)])
def test_scan_velocity_off_its_mirror_external(ctx, nw, group):
    """DerOmega with external terms on such channels, in groups of one band and of a few.  What the kernel reads
    as Hermitian is so in the reference: the product V D' of dD.nl = -(dD.ln)^+ (its within-group part has
    V''_nq D'_ql as stored), and the real part of dO.nn."""
    from oracle import wb_oracle as O
    from wannierberri_amd import _lib
    X, E, dEF, level, d = _off_mirror(nw, True, group)
    f = O.DerOmega(d)
    V, W, Dh, m = d.Xbar("Ham", 1), d.Xbar("Ham", 2), d.D_H, d.dEig_inv

    class DerD(O.DerDcov):
        def nl(self, ik, inn, out):
            pv = np.einsum("lpb,pnd->lnbd", V[ik][out][:, out], Dh[ik][out][:, inn])
            own = np.einsum("nqb,qld->lnbd", V[ik][inn][:, inn], Dh[ik][inn][:, out])
            s = (W[ik][out][:, inn] + pv + pv.swapaxes(2, 3)).conj() + own + own.swapaxes(2, 3)
            return (m[ik][out][:, inn][:, :, None, None] * s).swapaxes(0, 1)

    class DerO:   # the diagonal, which a trace reads
        def nn(self, ik, inn, out):
            o, do = d.Xbar("rotAA")[ik], d.Xbar("rotAA", 1)[ik]
            diag = (do[inn, inn] + 2 * np.einsum("lnc,lnd->ncd", o[out][:, inn].conj(), Dh[ik][out][:, inn])).real
            return np.eye(len(inn))[:, :, None, None] * diag[:, None]
    f.dD, f.dO = DerD(d), DerO()
    hist = _scan_bins(ctx, X, E, dEF, level, _lib.FORMULA_DEROMEGA, True)
    ref = np.zeros_like(hist)
    bands = np.arange(nw)
    for ik in range(len(E)):
        for g in np.unique(bands // group):
            inn = bands[bands // group == g]
            e = E[ik, inn].mean()
            ref[int(np.ceil(e / dEF))] += f.trace(ik, inn, np.delete(bands, inn)).reshape(9)
    err = np.abs(hist - ref).max() / np.abs(ref).max()
    print(f"test_scan_velocity_off_its_mirror_external nw={nw} group={group}: {err:.1e}", flush=True)
    assert err < 1e-12   # as above


@pytest.mark.parametrize("nw", [1, 2, 15, 16, 17, 31, 32, 33, 48, 49, 64, 65, 80, 81, 97, 112, 113, 128])
def test_rotate_sizes(ctx, nw):
    """One size at each edge of the rotation's 16-row blocks, flagged (Hermitian part), plain and
    skipped channels: sums of nw^2 products in FP64 (complex64: rounded once more on storing)."""
    import torch
    from wannierberri_amd import _lib
    rng = np.random.default_rng(nw)
    nk, nch = 3, 6
    U = np.linalg.qr(rng.standard_normal((nk, nw, nw)) + 1j * rng.standard_normal((nk, nw, nw)))[0]
    X = rng.standard_normal((nk, nch, nw, nw)) + 1j * rng.standard_normal((nk, nch, nw, nw))
    herm = np.array([0, 1, 1, 0, 0, 1], dtype=np.int32)
    skip = np.array([0, 0, 1, 0, 1, 0], dtype=np.int32)
    for prec, cd, nd, eps in ((_lib.WBMI_F64, torch.complex128, complex, EPS), (_lib.WBMI_F32, torch.complex64, np.complex64, 6e-8)):
        Us, Xs = U.astype(nd), X.astype(nd)
        Xd, Ud = torch.from_numpy(Xs).cuda(), torch.from_numpy(Us).cuda()
        ctx.rotate(Ud, Xd, herm, skip, prec)
        got = Xd.cpu().numpy()
        Uw, Xw = Us.astype(complex), Xs.astype(complex)
        Xw = np.where(herm[None, :, None, None] == 1, 0.5 * (Xw + Xw.conj().swapaxes(2, 3)), Xw)
        ref = Uw.conj().swapaxes(1, 2)[:, None] @ Xw @ Uw[:, None]
        ref = np.where(skip[None, :, None, None] == 1, Xs, ref)
        bound = 4 * EPS * nw * np.abs(X).max() * np.sqrt(nw) + (eps * np.abs(ref).max() if eps > EPS else 0)
        assert np.abs(got - ref).max() < bound


@pytest.mark.parametrize("nw", [2, 15, 16, 17, 29, 32])
def test_rotate_order_of_sums(ctx, nw):
    """complex64 channels: at most 32 bands are summed in the order in which more than 64 are (the summed index,
    four at a time), so that a rounding does not depend on the kernel that a size takes.  The matrices
    stand alone and in the corner of 70 x 70 ones; sums that cancel to 1e-10 of their terms show the order."""
    import torch
    from wannierberri_amd import _lib
    rng = np.random.default_rng(nw)
    nk, nch, big = 2, 5, 70
    def rand(*shape):
        return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)
    U = rand(nk, nw, nw)
    X = 1e10 * rand(nk, nch, nw, nw)
    pick = rng.permutation(nw)   # the terms of pairs (i, j) of the summed index cancel in the products
    for i, j in zip(pick[0::2], pick[1::2]):
        U[:, j] = U[:, i]
        X[:, :, :, j] = -X[:, :, :, i]
    X[:, :, :, pick[-1]] = rand(nk, nch, nw)
    Xb, Ub = np.zeros((nk, nch, big, big), np.complex64), np.zeros((nk, big, big), np.complex64)
    Xb[:, :, :nw, :nw], Ub[:, :nw, :nw] = X, U
    out = []
    for x, u in ((X, U), (Xb, Ub)):
        xd = torch.from_numpy(x.copy()).cuda()
        ctx.rotate(torch.from_numpy(u).cuda(), xd, None, None, _lib.WBMI_F32)
        out.append(xd.cpu().numpy()[:, :, :nw, :nw])
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("nk,nw,extra", [(1, 1, 0), (7, 3, 0), (17, 5, 1), (33, 4, 2), (130, 7, 1)])
def test_klist_pairs(ctx, nk, nw, extra):
    """R -> k with the R-vectors in pairs against the single-vector form and the plain sum: lists with
    R-vectors that lack their -R, a repeated vector, and numbers of pairs off the chunk size."""
    import torch
    from wannierberri_amd import _lib
    from wannierberri_amd.data_k import r_pairs
    rng = np.random.default_rng(nk)
    r = np.arange(-2, 3)
    iR = np.array([[x, y, z] for x in r for y in r for z in r[:3 + extra % 2]], dtype=np.int32)
    iR = np.concatenate([rng.permutation(iR), [[7, 0, -1]], iR[:extra]]).astype(np.int32)
    pairs = r_pairs(iR)
    flat = pairs.ravel()
    assert sorted(flat[flat >= 0]) == list(range(len(iR)))
    for i, j in pairs:
        assert j < 0 or (iR[i] == -iR[j]).all()
    nelem = 3 * nw * nw
    X = rng.standard_normal((len(iR), nelem)) + 1j * rng.standard_normal((len(iR), nelem))
    k = rng.random((nk, 3))
    ref = np.exp(2j * np.pi * (k @ iR.T)) @ X
    d = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()  # noqa: E731
    Xd, kd, iRd = d(X), d(k), d(iR)
    # phases are off by the rounding of k.R (|R| <= 8) times 2 pi
    bound = 2 * np.pi * 16 * EPS * np.abs(X).sum(axis=0).max()
    for prec, cd in ((_lib.WBMI_F64, torch.complex128), (_lib.WBMI_F32, torch.complex64)):
        out = torch.empty((nk, 3, nw, nw), dtype=cd, device="cuda")
        for tile in [None] + list(range(7)):
            for p in (None, d(pairs)):
                out.zero_()
                ctx.r2k_klist(iRd, Xd, kd, out, prec, tile=tile, pairs=p)
                err = np.abs(out.cpu().numpy().reshape(nk, nelem) - ref).max()
                assert err < bound + (1.2e-7 * np.abs(ref).max() if prec == _lib.WBMI_F32 else 0), (tile, p is None)


@pytest.mark.parametrize("nk,nelem", [(1, 64 * 65535 + 1), (17, 64 * 65535 + 1), (2, 128 * 65535)])
def test_klist_many_elements(ctx, nk, nelem):
    """More elements per k-point than the narrow tiles take: up to 128 x 65535 are accepted for any list."""
    import torch
    from wannierberri_amd import _lib
    iR = torch.tensor([[0, 0, 0], [1, 0, 0]], dtype=torch.int32, device="cuda")
    X = torch.ones((2, nelem), dtype=torch.complex128, device="cuda")
    X[1] = torch.linspace(0, 1, nelem, dtype=torch.float64, device="cuda")
    k = np.random.default_rng(nk).random((nk, 3))
    out = torch.zeros((nk, nelem), dtype=torch.complex128, device="cuda")
    ctx.r2k_klist(iR, X, torch.from_numpy(k).cuda(), out, _lib.WBMI_F64, tile=-1)
    ref = 1 + torch.from_numpy(np.exp(2j * np.pi * k[:, :1])).cuda() * X[1]
    assert (out - ref).abs().max().item() < 2 * np.pi * 4 * EPS * 2   # the phase's rounding, as in test_klist_pairs
    with pytest.raises(ValueError, match="elements per k-point"):
        ctx.r2k_klist(iR, torch.empty((2, 128 * 65535 + 1), dtype=torch.complex128, device="cuda"), torch.from_numpy(k).cuda(),
                      torch.empty((nk, 128 * 65535 + 1), dtype=torch.complex128, device="cuda"), _lib.WBMI_F64, tile=-1)


@pytest.mark.parametrize("ibands", [None, [4, 1, 2]])
def test_tables_under_way(monkeypatch, ibands):
    """Tabulated results over several blocks, their host copies at once or behind the queued work: the same
    numbers, as a result, as its pickle, per block and along a path."""
    import pickle
    import wannierberri_amd as wb
    from wannierberri_amd import models
    from wannierberri_amd.result import HostCopy
    tab = wb.calculators.tabulate
    s = models.synthetic(num_wann=5, Rmax=1, seed=8)
    path = wb.Path(system=s, k_list=np.linspace([0, 0, 0], [0.5, 0.4, 0.1], 12))
    grid = wb.Grid(system=s, NK=[4, 4, 2], NKFFT=[2, 2, 2])
    out = []
    for limit in (0, 1 << 30):
        monkeypatch.setattr(HostCopy, "LIMIT", limit)
        r = []
        for g, kw in ((path, {"k_batch": 5}), (grid, {"symmetrize": False, "use_irred_kpt": False})):
            t = tab.TabulatorAll({"Energy": tab.Energy(), "vel": tab.Velocity(), "berry": tab.BerryCurvature()}, ibands=ibands,
                                 mode="path" if g is path else "grid")
            res = wb.run(s, g, {"t": t}, save_files=False, verbose=False, **kw).results["t"].results
            r += [res[k].data for k in ("Energy", "vel", "berry")] + [pickle.loads(pickle.dumps(res["berry"])).data]
        block = tab.BerryCurvature(ibands=ibands)
        from wannierberri_amd.data_k import Data_K
        one = [block(Data_K(s, k_list=[[0.1 * i, 0.2, 0.3], [0.4, 0.1, 0.1 * i]])) for i in range(3)]
        total = one[0] + one[1] + one[2]
        r += [total.data] + [x.data for x in one]
        assert np.array_equal(total.data, np.concatenate([x.data for x in one]))
        out.append(r)
    for a, b in zip(*out):
        assert a.shape == b.shape and a.shape[1] == (5 if ibands is None else 3)
        # (the traces' partial sums meet in any order)
        assert np.abs(a - b).max() < 1e-12 * np.abs(a).max()


def test_klist_pairs_on_demand(ctx, monkeypatch):
    """A grid never forms the pairs (R, -R); the first k-list does, once; while a graph capture is the first,
    the transform takes every R-vector alone."""
    import torch
    import wannierberri_amd as wb
    from wannierberri_amd import data_k, models
    formed = []
    real = data_k.r_pairs
    monkeypatch.setattr(data_k, "r_pairs", lambda R: formed.append(len(R)) or real(R))
    Ef = np.linspace(-4, 4, 9)
    k = np.random.default_rng(1).random((8, 3))
    calcs = {"ahc": wb.calculators.static.AHC(Efermi=Ef)}
    s = models.synthetic(num_wann=4, Rmax=1, seed=3)
    wb.run(s, wb.Grid(system=s, NK=[4, 4, 4], NKFFT=[4, 4, 4]), calcs, save_files=False, verbose=False)
    assert formed == []
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    alone = wb.run_klists(s, [k], calcs).results["ahc"].data
    assert formed == []
    monkeypatch.undo()
    monkeypatch.setattr(data_k, "r_pairs", lambda R: formed.append(len(R)) or real(R))
    for _ in range(2):
        pairs = wb.run_klists(s, [k], calcs).results["ahc"].data
    assert formed == [s.rvec.nRvec]
    # the phases' rounding (test_klist_pairs) over gaps of order one
    assert np.abs(alone - pairs).max() < 1e-11 * np.abs(pairs).max()


@pytest.mark.parametrize("nw,limit,nc", [(5, "k", 1), (5, "k", 3), (5, "bytes", 3), (66, "bytes", 3), (66, "bytes", 1)])
def test_corner_batches(monkeypatch, nw, limit, nc):
    """Corner energies in batches of one and three of the eight corners (the last batch not full), the batch
    limited by its k-points or by its memory (Hamiltonians, vectors and, above 64 bands, the eigensolver's
    workspace): the same energies as all corners together, no call beyond the limit."""
    import wannierberri_amd as wb
    from wannierberri_amd import _lib, data_k, models
    s = models.synthetic(num_wann=nw, Rmax=1, seed=nw)
    grid = wb.Grid(system=s, NK=[3, 3, 2], NKFFT=[3, 3, 2])
    Kp = grid.get_K_list(use_symmetry=False)[0]
    nk = 18

    def corners():
        return data_k.Data_K(s, dK=Kp.Kp_fullBZ, grid=grid, Kpoint=Kp).corner_energies().cpu().numpy()
    ref = corners()
    per_corner = nk * nw * nw * 16 * (2 + (4 if nw > 64 else 0))
    if limit == "k":
        monkeypatch.setattr(data_k, "CORNER_BATCH_K", nc * nk + 1)
    else:
        monkeypatch.setattr(data_k, "CORNER_BATCH_BYTES", nc * per_corner + 1)
    calls = []
    eigh = _lib.Context.eigh
    monkeypatch.setattr(_lib.Context, "eigh", lambda self, H, st, E, *a, **k: calls.append(len(E)) or eigh(self, H, st, E, *a, **k))
    got = corners()
    assert calls[1:] == [nc * nk] * (8 // nc) + ([8 % nc * nk] if 8 % nc else [])   # [0]: the block itself
    assert np.abs(got - ref).max() < 8 * EPS * nw * np.abs(ref).max()


@pytest.mark.parametrize("nw,nef,nom,kbt,smr", [(2, 1, 1, 0.0, "Lorentzian"), (5, 8, 16, 0.05, "Gaussian"), (6, 15, 17, 0.0, "Lorentzian"),
                                                (9, 7, 129, 0.05, "Lorentzian"), (20, 3, 128, 0.05, "Lorentzian"),
                                                (34, 2, 3, 0.05, "Lorentzian")])
def test_optical_tiles(ctx, nw, nef, nom, kbt, smr):
    """Optical conductivity at the edges of its output tiles (128 frequencies, 64 columns of (Fermi level,
    component)), of the pair batches and of the LDS form, with a pair of bands in one group, vs the oracle."""
    import wannierberri_amd as wb
    from oracle import wb_oracle as O
    from wannierberri_amd import models
    s = models.synthetic(num_wann=nw, Rmax=1, seed=70 + nw)
    ham = s.get_R_mat("Ham").copy()
    if nw > 4:
        ham[:, -2:, :] = 0.
        ham[:, :, -2:] = 0.
        ham[s.rvec.iR0, -2, -2], ham[s.rvec.iR0, -1, -1] = 0.3, 0.3 + 5e-5
        s.set_R_mat("Ham", ham, reset=True)
    Ef, om = np.linspace(-0.5, 0.5, nef), np.linspace(0.0, 4.0, nom)
    k = np.random.default_rng(nw).random((5, 3))
    kw = dict(kBT=kbt, smr_fixed_width=0.1, smr_type=smr)
    got = wb.run_klists(s, [k], {"opt": wb.calculators.dynamic.OpticalConductivity(Efermi=Ef, omega=om, **kw)})
    o = O.OracleSystem(s.real_lattice, s.rvec.iRvec, s.wannier_centers_cart, {m: s.get_R_mat(m) for m in ("Ham", "AA")})
    ref = O.OpticalConductivity(Ef, om, **kw)(O.OracleDataK(o, k_list=k)).data
    scale = np.abs(ref).max()
    if scale == 0:
        assert np.abs(got.results["opt"].data).max() == 0
    else:
        assert np.abs(got.results["opt"].data - ref).max() < 1e-10 * scale


@pytest.mark.parametrize("nw", [4, 34])
def test_optical_pairs_left_alone(ctx, nw):
    """A matrix element that is not finite is seen at the Fermi levels that part its two bands only."""
    import wannierberri_amd as wb
    from wannierberri_amd import models
    from wannierberri_amd.data_k import Data_K
    s = models.synthetic(num_wann=nw, Rmax=1, seed=nw)
    data = Data_K(s, k_list=[[0.1, 0.2, 0.3]], channels={("Ham", 1), ("AA", 0)})
    E = data.E_K[0]
    Ef = [E[0] - 1.0, 0.5 * (E[0] + E[1]), 0.5 * (E[1] + E[2]), 0.5 * (E[2] + E[3]), E[-1] + 1.0]
    calc = wb.calculators.dynamic.OpticalConductivity(Efermi=Ef, omega=np.linspace(0.0, 2.0, 5), kBT=0.0, smr_fixed_width=0.1)
    data.ensure(calc.needed_channels(s))
    for sl in data._slots.values():
        data.Xk[0, sl:sl + 3, 0, 1] = data.Xk[0, sl:sl + 3, 1, 0] = 0.0
    ref = calc(data).data
    sl = data._slots["Ham", 1]
    data.Xk[0, sl:sl + 3, 0, 1] = float("nan")
    got = calc(data).data
    assert np.isnan(got[1]).any()
    others = [0, 2, 3, 4]
    assert np.abs(got[others] - ref[others]).max() <= 1e-13 * np.abs(ref).max()
