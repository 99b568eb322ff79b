"""What a k-list transform needs on the device (no GPU): a k-list is copied without waiting only where the
stream orders it before its use; the R-vectors as pairs (R, -R)."""
import types

import numpy as np
import pytest

from wannierberri_amd.data_k import Data_K, r_pairs


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


@pytest.mark.parametrize("kind", ["ordered", "permuted", "without some -R", "repeated", "one", "far"])
def test_r_pairs(kind):
    """Every R-vector in one pair, partners opposite, none left alone that has a free partner."""
    rng = np.random.default_rng(3)
    r = np.arange(-2, 3)
    R = np.array([[x, y, z] for x in r for y in r for z in r], dtype=np.int32)
    R = {"ordered": R, "permuted": rng.permutation(R), "without some -R": rng.permutation(R)[:77],
         "repeated": np.concatenate([R[10:], R[:90]]), "one": R[:1], "far": R * 1000000}[kind].astype(np.int32)
    pairs = r_pairs(R)
    assert pairs.dtype == np.int32
    flat = pairs.ravel()
    assert sorted(flat[flat >= 0]) == list(range(len(R))) and (pairs[:, 0] >= 0).all()
    assert all(j < 0 or (R[i] == -R[j]).all() for i, j in pairs)
    alone = [tuple(R[i]) for i, j in pairs if j < 0]
    assert all(tuple(-x for x in a) not in alone for a in alone if any(a)) and alone.count((0, 0, 0)) <= 1
