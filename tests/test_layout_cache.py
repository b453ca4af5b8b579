"""The differentiable SpMM's cached block structures, on the host alone."""

import threading

import torch

from void_amd import _runtime, autograd


def test_record_once(monkeypatch):
    """An array is recorded on every stream that uses it, once each."""
    now, log = [7], []

    class Array:
        def __init__(self, name):
            self.name = name

        def record_stream(self, s):
            log.append((self.name, s))

    monkeypatch.setattr(_runtime, "raw_stream", lambda d: now[0])
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: now[0])
    seen = set()
    arrays = Array("a"), Array("b")
    for s in (7, 9, 7, 9):
        now[0] = s
        _runtime.record_once(seen, torch.device("cpu"), *arrays)
    assert log == [("a", 7), ("b", 7), ("a", 9), ("b", 9)]


def test_layout_lookup_from_threads(monkeypatch):
    """Threads that overflow the cache at the same time: every look-up gives its
    own structure's order, and none raises."""
    monkeypatch.setattr(autograd, "_LAYOUTS", {})
    errors = []

    def work(k):
        try:
            g = torch.Generator().manual_seed(k)
            for _ in range(150):
                flat = torch.randperm(48, generator=g)[:9]
                rows, cols = (flat // 8).int(), (flat % 8).int()
                lay = autograd._layout(rows, cols, (192, 256))
                assert torch.equal(lay.order, torch.argsort(flat, stable=True))
        except Exception as e:
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
