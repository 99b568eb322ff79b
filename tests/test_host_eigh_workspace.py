"""Which sizes of the refined eigensolver ask for a workspace (no GPU calls)."""
import pytest

from wannierberri_amd import _lib


@pytest.mark.parametrize("nw", [1, 32, 44, 45, 64, 65, 128])
def test_eigh_work_bytes(nw):
    """Up to 64 bands the refinement keeps its matrices in LDS and registers; above, four FP64 complex
    matrices per k-point."""
    for prec in (_lib.WBMI_F64, _lib.WBMI_F32):
        assert _lib.lib().wbmi_eigh_work_bytes(300, nw, prec, 16) == (4 * 16 * nw * nw * 300 if nw > 64 else 0)
        assert _lib.lib().wbmi_eigh_work_bytes(300, nw, prec, 0) == 0
