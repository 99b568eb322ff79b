"""A k-list goes to the device without waiting only where the stream orders it before its use (no GPU)."""
import types

import numpy as np
import pytest

from wannierberri_amd.data_k import Data_K


@pytest.mark.parametrize("own,idle", [(True, True), (True, False), (False, True), (False, False)])
def test_klist_copy(own, idle):
    """`own`: torch's current stream is the one the transform runs on; `idle`: nothing is queued there."""
    done = []

    class Host:
        pinned = False

        def pin_memory(self):
            h = Host()
            h.pinned = True
            return h

        def to(self, device, non_blocking=False):
            done.append((self.pinned, non_blocking))
            return "on the device"
    stream = types.SimpleNamespace(query=lambda: idle)
    torch = types.SimpleNamespace(from_numpy=lambda a: Host(), empty=lambda *a, **k: "out", cuda=types.SimpleNamespace(
        current_stream=lambda device=None: stream if own else "another stream"))
    d = object.__new__(Data_K)
    d.torch, d.num_wann, d.nk, d.k_list, d.k_list_dev, d._pref = torch, 2, 3, np.zeros((3, 3)), None, None
    d.dev = types.SimpleNamespace(stack=lambda keys: np.zeros((1, 1, 2, 2)), iRvec_dev=None, pairs_dev=None)
    used = []
    d.ctx = types.SimpleNamespace(stream=stream, device="gpu", r2k_klist=lambda iR, X, kl, out, prec, pairs: used.append(kl))
    d._transform([("Ham", 0)], None, 0)
    ahead = own and not idle
    assert done == [(ahead, ahead)] and used == ["on the device"]
