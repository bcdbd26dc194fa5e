"""The buffers a context keeps between calls (hit records, rows of gradient sums), without a GPU: stand-ins for tensors,
streams and events that note what is asked of them."""
import pytest
import torch

from diff_surfel_tracing import _C


class _Stream:
    def __init__(self):
        self.waited = []

    def wait_event(self, event):
        self.waited.append(event)


class _Event:
    def record(self, stream):
        self.stream = stream


class _Buffer:
    """A device tensor as the caching allocator sees it: `home` is the stream it was made on, `users` the streams the
    allocator has been told of.  Once it is dropped the memory is free for `home` as soon as those are done with it."""

    def __init__(self, n, dtype, device, home):
        self.n, self.dtype, self.device, self.home, self.users, self.is_cuda = n, dtype, device, home, [], True

    def numel(self):
        return self.n

    def element_size(self):
        return {torch.float32: 4, torch.int64: 8, torch.uint8: 1}[self.dtype]

    def record_stream(self, stream):
        if stream is not self.home:
            self.users.append(stream)


class _Device:
    """What the pools ask of torch.cuda, with a current stream that the test sets."""

    def __init__(self, monkeypatch):
        self.now, self.capturing = _Stream(), False
        make = lambda n, dtype=torch.float32, device=None: _Buffer(n, dtype, device, self.now)  # noqa: E731
        monkeypatch.setattr(_C, "_current_stream", lambda: self.now)
        monkeypatch.setattr(_C.torch.cuda, "Event", _Event)
        monkeypatch.setattr(_C.torch.cuda, "current_device", lambda: 0)
        monkeypatch.setattr(_C.torch.cuda, "is_current_stream_capturing", lambda: self.capturing)
        monkeypatch.setattr(_C.torch, "zeros", make)
        monkeypatch.setattr(_C.torch, "empty", make)


@pytest.fixture
def device(monkeypatch):
    return _Device(monkeypatch)


def _context():
    ctx = _C.OptiXStateWrapper.__new__(_C.OptiXStateWrapper)
    ctx.handle = None
    ctx._row_pool, ctx._record_pool, ctx._record_fixed, ctx._record_events, ctx._record_watch = [], [], False, {}, []
    ctx.record_blocks_per_wave, ctx.deterministic, ctx.records_skipped = 4.0, False, 0
    ctx.record_max_bytes, ctx.record_pool_max_bytes, ctx.row_pool_max_bytes = 1 << 40, 1 << 40, 1 << 40
    return ctx


def test_gradient_rows_tell_the_allocator_of_every_stream_they_serve(device):
    """A pair made on one stream and used on another may be dropped while that other one still works on it (P grew, the
    mode changed, the tracer went away): the allocator has to know."""
    ctx = _context()
    a, b = device.now, _Stream()
    pair = ctx.acquire_rows(10, 660, torch.float32, "cuda:0")
    ctx.release_rows(*pair)
    device.now = b
    again = ctx.acquire_rows(10, 660, torch.float32, "cuda:0")
    assert again[0] is pair[0] and again[1] is pair[1]
    assert len(b.waited) == 1 and b.waited[0].stream is a
    assert pair[0].users == [b] and pair[1].users == [b]
    ctx.release_rows(*again)
    device.now = a                              # and back: nothing new to be told of, but b has to be waited for
    assert ctx.acquire_rows(10, 660, torch.float32, "cuda:0")[0] is pair[0]
    assert a.waited[-1].stream is b and pair[0].users == [b]


class _Record:
    """HitRecord without the library behind it."""

    def __init__(self, H, W, mtd_alloc, blocks_per_wave, device, storage=None):
        self.words, self.blocks = storage, 1

    @classmethod
    def layout(cls, H, W, mtd_alloc, blocks_per_wave):
        return H * W, 4, 1, 1


def test_hit_records_tell_the_allocator_of_every_stream_they_serve(device, monkeypatch):
    monkeypatch.setattr(_C, "HitRecord", _Record)
    ctx = _context()
    a, b, c = device.now, _Stream(), _Stream()
    rec = ctx.acquire_record(8, 8, 1, torch.device("cuda", 0))
    storage = rec.words
    ctx.release_record(rec)
    device.now = b                              # a forward trace there, whose graph may go without a backward pass
    rec = ctx.acquire_record(8, 8, 1, torch.device("cuda", 0))
    assert rec.words is storage and b.waited[0].stream is a and storage.users == [b]
    device.now = c                              # a backward trace on a stream of its own
    ctx.release_record(rec)
    assert c in storage.users


def _held(ctx):
    return sum(r.n * r.element_size() + m.n for r, m, _, _ in ctx._row_pool)


def test_gradient_rows_kept_between_calls_are_bounded_and_given_back(device):
    ctx = _context()
    pairs = [ctx.acquire_rows(10, 660, torch.float32, "cuda:0") for _ in range(3)]
    assert len({id(p[0]) for p in pairs}) == 3
    one = 4 * 660 + 10
    for p in pairs:
        ctx.release_rows(*p)
    assert _held(ctx) == 2 * one                       # ROW_POOL_SIZE pairs
    ctx.row_pool_max_bytes = 2 * one - 1
    ctx.release_rows(*ctx.acquire_rows(10, 660, torch.float32, "cuda:0"))
    assert _held(ctx) == one                           # and a limit in bytes
    # the mode changed, or the scene grew: what no longer fits is not held beside what does
    det = ctx.acquire_rows(10, 660, torch.int64, "cuda:0")
    assert _held(ctx) == 0
    ctx.row_pool_max_bytes = 8 * 660
    ctx.release_rows(*det)
    assert _held(ctx) == 0                             # 8 * 660 + 10: more than the limit, not kept at all
    ctx.row_pool_max_bytes = 1 << 30
    ctx.release_rows(*ctx.acquire_rows(10, 660, torch.int64, "cuda:0"))
    grown = ctx.acquire_rows(20, 1320, torch.int64, "cuda:0")
    assert _held(ctx) == 0
    ctx.release_rows(*grown)
    assert ctx.acquire_rows(10, 660, torch.int64, "cuda:0")[0] is grown[0]   # larger than needed: serves
    ctx.release_rows(*grown)

    class _Pending:                                    # a forward trace that nobody traced backward through
        def asked(self, wait=False):
            return None
    ctx._record_watch.append(_Pending())
    ctx.release_memory()
    assert _held(ctx) == 0 and not ctx._record_watch


def test_threads_never_share_a_buffer(device, monkeypatch):
    """Several threads that draw from one context's pools and give back: nobody holds what somebody else holds."""
    import sys
    import threading
    monkeypatch.setattr(_C, "HitRecord", _Record)
    ctx = _context()
    held, clashes, guard = set(), [], threading.Lock()

    def hold(*buffers):
        with guard:
            clashes.extend(b for b in buffers if id(b) in held)
            held.update(id(b) for b in buffers)

    def let_go(*buffers):
        with guard:
            held.difference_update(id(b) for b in buffers)

    def work():
        for _ in range(3000):
            rows, marks = ctx.acquire_rows(4, 264, torch.float32, torch.device("cuda", 0))
            rec = ctx.acquire_record(8, 8, 1, torch.device("cuda", 0))
            words = rec.words
            hold(rows, marks, words)
            let_go(rows, marks, words)
            ctx.release_rows(rows, marks)
            ctx.release_record(rec)
    interval = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)
    try:
        threads = [threading.Thread(target=work) for _ in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(interval)
    assert not clashes
    assert len(ctx._record_pool) <= ctx.RECORD_POOL_SIZE and len(ctx._record_events) <= ctx.RECORD_POOL_SIZE


def test_a_captured_step_keeps_its_buffers_to_itself(device, monkeypatch):
    """A graph writes to the same memory on every replay: what a captured call takes is its own, not the pool's, and does
    not go on to other calls."""
    monkeypatch.setattr(_C, "HitRecord", _Record)
    ctx = _context()
    dev = torch.device("cuda", 0)
    rec, pair = ctx.acquire_record(8, 8, 1, dev), ctx.acquire_rows(10, 660, torch.float32, dev)
    pooled = [rec.words, pair[0], pair[1]]
    ctx.release_record(rec)
    ctx.release_rows(*pair)
    device.capturing = True
    rec, pair = ctx.acquire_record(8, 8, 1, dev), ctx.acquire_rows(10, 660, torch.float32, dev)
    taken = [rec.words, pair[0], pair[1]]
    assert not any(t is p for t in taken for p in pooled)
    ctx.release_record(rec)
    ctx.release_rows(*pair)
    assert rec.words is None
    device.capturing = False
    rec, pair = ctx.acquire_record(8, 8, 1, dev), ctx.acquire_rows(10, 660, torch.float32, dev)
    assert [rec.words, pair[0], pair[1]] == pooled
    rec, pair = ctx.acquire_record(8, 8, 1, dev), ctx.acquire_rows(10, 660, torch.float32, dev)
    assert not any(t is x for t in (rec.words, *pair) for x in taken)
