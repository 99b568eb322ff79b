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
