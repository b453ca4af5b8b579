"""The differentiable SpMM's cached block structures, on the host alone."""

import copy
import io
import threading
import weakref
from collections import OrderedDict

import pytest
import torch

import void_amd
from void_amd import _runtime, _streams, autograd


def test_record_once(monkeypatch):
    """An array is recorded on every stream that uses it, once each."""
    now, log = [7], []

    class Array:
        def __init__(self, name):
            self.name = name

        def record_stream(self, s):
            log.append((self.name, s))

    monkeypatch.setattr(_streams, "raw_stream", lambda d: now[0])
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: now[0])
    seen = set()
    arrays = Array("a"), Array("b")
    for s in (7, 9, 7, 9):
        now[0] = s
        _streams.record_once(seen, torch.device("cpu"), *arrays)
    assert log == [("a", 7), ("b", 7), ("a", 9), ("b", 9)]


@pytest.fixture
def cache(monkeypatch):
    """The cache, empty, and a list of the layouts that are built."""
    monkeypatch.setattr(autograd, "_ALIVE", weakref.WeakValueDictionary())
    monkeypatch.setattr(autograd, "_RECENT", OrderedDict())
    monkeypatch.setattr(autograd, "_OWNED", weakref.WeakKeyDictionary())
    built = []
    build = autograd.build_bsr_layout
    monkeypatch.setattr(autograd, "build_bsr_layout", lambda *a: built.append(a) or build(*a))
    return built


def _index(seed, n=9):
    flat = torch.randperm(48, generator=torch.Generator().manual_seed(seed))[:n]
    return flat, (flat // 8).int(), (flat % 8).int()


def test_layout_lookup_from_threads(cache):
    """Threads that overflow the cache at the same time: every look-up gives its
    own structure's order, and none raises."""
    errors = []

    def work(k):
        try:
            for i in range(150):
                flat, rows, cols = _index(1000 * k + i)
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
    assert len(autograd._RECENT) == autograd.MAX_RECENT == len(autograd._ALIVE)


def test_modules_keep_their_structures(cache):
    """More modules than the list of recent structures is long: the second round
    over them builds nothing, and a module's end frees what it kept."""
    mods = [torch.nn.Identity() for _ in range(3 * autograd.MAX_RECENT)]
    index = [_index(i)[1:] for i in range(len(mods))]
    for _ in range(2):
        for m, (rows, cols) in zip(mods, index):
            s = autograd._structure(rows, cols, (192, 256), m)
            assert s.transposed is s.transposed
        assert len(cache) == 2 * len(mods)
    for m, (rows, cols) in zip(mods, index):  # the bare function finds them too
        assert autograd._structure(rows, cols, (192, 256)) is autograd._OWNED[m]
    assert len(cache) == 2 * len(mods)
    autograd._RECENT.clear()
    del s, m
    mods.clear()
    assert len(autograd._ALIVE) == 0 == len(autograd._OWNED)


def test_bare_structures_leave_one_by_one(cache):
    index = [_index(i)[1:] for i in range(autograd.MAX_RECENT + 1)]
    for rows, cols in index:
        autograd._layout(rows, cols, (192, 256))
    for rows, cols in index[1:]:
        autograd._layout(rows, cols, (192, 256))
    assert len(cache) == len(index)


def test_structure_key(cache):
    """Changed in place, or another view of the same memory: another structure."""
    _, rows, cols = _index(3, 8)
    first = autograd._layout(rows, cols, (192, 256))
    assert autograd._layout(rows, cols, (192, 256)) is first
    assert autograd._layout(rows[::2], cols[::2], (192, 256)) is not autograd._layout(rows[:4], cols[:4], (192, 256))
    rows[0] = (rows[0] + 1) % 6
    assert autograd._layout(rows, cols, (192, 256)) is not first


def test_modules_copy_and_pickle():
    """A module that has kept a structure is copied and stored as before."""
    _, rows, cols = _index(5)
    vt = void_amd.VOIDTensor(values=torch.randn(9, 32, 32), block_rows=rows, block_cols=cols,
                             morton_codes=torch.zeros(9, dtype=torch.int64), shape=(192, 256), tile_size=(32, 32),
                             nnz_original=0, n_blocks=9, density=0.0)
    lin = void_amd.SparseLinear(256, 192, vt)
    autograd._structure(lin.sparse_weight.block_rows, lin.sparse_weight.block_cols, (192, 256), lin.sparse_weight)
    buf = io.BytesIO()
    torch.save(lin, buf)
    buf.seek(0)
    for other in (copy.deepcopy(lin), torch.load(buf, weights_only=False)):
        assert torch.equal(other.sparse_weight.values, lin.sparse_weight.values)
        assert other.sparse_weight not in autograd._OWNED


def test_stream_workspaces(monkeypatch):
    """Plans of one stream share a buffer: counters are zero on entry whatever
    the plan before wrote as partials; large ones are not kept; streams are bounded."""
    monkeypatch.setattr(_runtime, "_zero_on_stream", lambda t, s, d: t.zero_())
    monkeypatch.setattr(_runtime, "MAX_SPARE_WORKSPACE", 1 << 16)
    pool, dev = _runtime.StreamWorkspaces(), torch.device("cpu")
    g = torch.Generator().manual_seed(0)
    for _ in range(200):
        counters = 256 * int(torch.randint(1, 9, (1,), generator=g))
        nbytes = counters + 256 * int(torch.randint(1, 300, (1,), generator=g))
        ws = pool.take(counters, nbytes, dev, int(torch.randint(0, 3, (1,), generator=g)))
        assert ws.numel() >= nbytes and not ws[:counters].any()
        ws[counters:nbytes] = 1  # a launch writes its partials and leaves the counters at zero
        assert all(b.numel() <= 1 << 16 for b, _ in pool.buffers.values())
    assert len(pool.buffers) == 3
    for stream in range(20):
        pool.take(256, 1024, dev, stream)
    assert list(pool.buffers) == [(dev, s) for s in range(12, 20)]
