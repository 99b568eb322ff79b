"""KBandResult: sums hold arrays of their own, whatever was read before or is changed after; shapes are
checked at the sum; pickles, threads."""
import copy
import pickle
import threading

import numpy as np
import pytest

from wannierberri_amd.result import HostCopy, KBandResult


@pytest.fixture
def now(monkeypatch):
    monkeypatch.setattr(HostCopy, "LIMIT", 0)   # copied at once: no GPU needed

    def make(a):
        import torch
        return KBandResult(HostCopy(torch.from_numpy(a), lambda x: x * 2.0, a.shape), 1, -1)
    return make


def test_sum_does_not_share(now):
    a0, b0 = np.arange(12.).reshape(2, 6), np.arange(6.).reshape(1, 6)
    for given in (False, True):
        for read in (False, True):
            a, b = (KBandResult(a0 * 2), KBandResult(b0 * 2)) if given else (now(a0), now(b0))
            want = np.concatenate([a0, b0]) * 2
            held = (a.data, b.data) if read else ()
            c, d = a + b, a + b
            for x in held:
                x[...] = -1.0
            a.data[...] = -2.0
            b.data *= 3.0
            c.data[0] += 1.0
            assert np.array_equal(d.data, want) and np.array_equal(c.data[1:], want[1:])
            assert c.data is c.data and c.nk == 3 and c.nband == 6 and c.rank == 0
    a = now(a0)
    e = a + 0
    assert e is a and np.array_equal(a.data, a0 * 2)


def test_sum_checks_shapes(now):
    a = now(np.zeros((2, 3)))
    for other in (np.zeros((2, 4)), np.zeros((2, 3, 3))):
        with pytest.raises(ValueError):
            a + now(other)
        with pytest.raises(ValueError):
            a + KBandResult(other)

    class Duck:
        data = np.ones((1, 3))
    assert np.array_equal((a + Duck()).data, [[0] * 3, [0] * 3, [1] * 3])


def test_pickle_and_copy(now):
    a0 = np.arange(6.).reshape(2, 3)
    s = now(a0) + now(a0)
    for r in (pickle.loads(pickle.dumps(s)), copy.deepcopy(s)):
        assert np.array_equal(r.data, np.concatenate([a0, a0]) * 2) and (r.transformTR, r.transformInv) == (1, -1)
        assert np.array_equal((r + now(a0)).data[4:], a0 * 2)
    # the state a pickle has always held
    assert set(s.__getstate__()) == {"data", "transformTR", "transformInv"}
    old = KBandResult.__new__(KBandResult)
    old.__setstate__({"data": a0, "transformTR": None, "transformInv": None})
    assert old.data is a0 and old.nk == 2


def test_threads(monkeypatch):
    """Threads that read one result and its sums while its copy is under way see the same arrays."""
    import time
    import torch

    class Event:
        def record(self, stream):
            pass

        def synchronize(self):
            time.sleep(1e-3)
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: None)

    def under_way():
        def finish(a):
            time.sleep(1e-3)
            return a * 2.0
        return KBandResult(HostCopy(torch.ones((4, 3)), finish, (4, 3)))
    for _ in range(20):
        a, b = under_way(), under_way()
        c = a + b
        out, start = [], threading.Barrier(9)

        def read(r):
            start.wait()
            out.append((r, r.data))
        ts = [threading.Thread(target=read, args=(r,)) for r in (a, c, b) * 3]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert len(out) == 9 and all(r.data is x and (x == 2).all() for r, x in out)
