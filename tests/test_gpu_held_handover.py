"""A buffer of the library's workspace pool that changes hands while its last owner's launches are still
running: whoever takes it over runs behind them (the two with operands and results of their own), and
the call that takes it over returns at once, whatever the device is doing."""
import contextlib

import pytest
import torch

from adrastea_amd import _ffi

pytestmark = pytest.mark.gpu

MIB = 1 << 20
SMALL = (128, 11008, 4096)   # rows, K, N: split along K in a buffer of 16 MiB
BIG = (640, 22016, 4096)     # ... that does not fit one


@pytest.fixture
def pool():
    lib = _ffi.lib()
    torch.cuda.synchronize()
    assert lib.adr_release_held_workspace_all() == 0
    lib.adr_set_held_workspace_limit(_ffi.HELD_WORKSPACE_DEFAULT_BYTES)
    yield lib
    lib.adr_set_held_workspace_limit(0)
    torch.cuda.synchronize()
    assert lib.adr_release_held_workspace_all() == 0


class Product:
    """x[M, K] . w[N, K]^T with operands of its own; `want` comes from the entry point with a workspace
    argument, whose sums are in the same order."""

    def __init__(self, lib, size, seed):
        self.lib, self.size = lib, size
        m, k, n = size
        g = torch.Generator(device="cuda").manual_seed(seed)
        self.x = torch.randn(m, k, dtype=torch.float16, device="cuda", generator=g)
        self.w = torch.randn(n, k, dtype=torch.float16, device="cuda", generator=g) * k ** -0.5
        self.out, self.want = (torch.zeros(m, n, dtype=torch.float16, device="cuda") for _ in range(2))
        need = lib.adr_matmul_f16_workspace_bytes(1, m, k, n, 1, n, 0, 1, k, 0, k, 1, 0, 0, 0, 0)
        assert (need > 16 * MIB) == (size == BIG) and need > 0
        room = 16 * MIB if size == SMALL else need
        ws = torch.empty(room, dtype=torch.uint8, device="cuda")
        assert lib.adr_matmul_f16_ws(torch.cuda.current_stream().cuda_stream, *self.args(self.want), ws.data_ptr(),
                                     room) == 0
        torch.cuda.synchronize()

    def args(self, out):
        m, k, n = self.size
        return (out.data_ptr(), self.x.data_ptr(), self.w.data_ptr(), 1, m, k, n, 1, n, 0, 1, k, 0, k, 1, 0, None,
                0.0, 1.0, 0, 0, 0)

    def run(self, stream):
        assert self.lib.adr_matmul_f16(stream.cuda_stream, *self.args(self.out)) == 0

    def right(self):
        return torch.equal(self.out.view(torch.int16), self.want.view(torch.int16))


class Load:
    """Some 40 ms of work for a stream to be busy with."""

    def __init__(self):
        self.a = torch.zeros(8192, 8192, dtype=torch.float16, device="cuda")
        self.b = torch.empty_like(self.a)
        torch.mm(self.a, self.a, out=self.b)   # (whatever the first call prepares)
        torch.cuda.synchronize()

    def put(self, stream):
        with torch.cuda.stream(stream):
            for _ in range(40):
                torch.mm(self.a, self.a, out=self.b)


def mark(stream):
    e = torch.cuda.Event(enable_timing=True)
    e.record(stream)
    return e


def streams(count):
    s = [torch.cuda.Stream() for _ in range(count)]
    assert len({x.cuda_stream for x in s}) == count
    return s


def independent(load, busy, candidates):
    """A stream that does not share a hardware queue with `busy` (it would run behind it in any case)."""
    for s in candidates:
        load.put(busy)
        behind, free = mark(busy), mark(s)
        torch.cuda.synchronize()
        if behind.elapsed_time(free) < 0:
            return s
    raise AssertionError("every stream shares the busy one's queue")


def test_a_call_that_takes_a_buffer_over_does_not_wait_for_the_device(pool):
    load, s = Load(), streams(17)
    products = [Product(pool, SMALL, 20 + i) for i in range(4)]
    for i in range(16):                       # s[0] has the pool to itself at first
        products[i % 3].run(s[i])
        torch.cuda.synchronize()
    assert pool.adr_held_workspace_bytes() == 16 * 16 * MIB
    declined = pool.adr_held_workspace_declined()
    load.put(s[0])
    busy = mark(s[0])
    products[3].run(s[16])
    assert not busy.query()                   # the call is back, the device still at work
    torch.cuda.synchronize()
    assert pool.adr_held_workspace_declined() == declined
    assert pool.adr_held_workspace_bytes() == 16 * 16 * MIB
    assert all(p.right() for p in products)


def test_the_least_recently_used_buffer_is_handed_on_in_order(pool):
    """The first takeover once all entries are taken, and one after it."""
    load, s = Load(), streams(21)
    one, other, rest = (Product(pool, SMALL, 30 + i) for i in range(3))

    def handed_on(owner, others, taker):
        one.out.zero_(), other.out.zero_()
        torch.cuda.synchronize()
        load.put(owner)
        one.run(owner)
        done = mark(owner)
        for x in others:                      # later than the owner's use
            rest.run(x)
        start = mark(taker)
        other.run(taker)
        end = mark(taker)
        running = not done.query()
        assert pool.adr_held_workspace_bytes() == 16 * 16 * MIB
        torch.cuda.synchronize()
        assert running and done.elapsed_time(start) < 0   # (the taker was free to begin before the owner was done)
        assert done.elapsed_time(end) > 0                 # its product waited
        assert one.right() and other.right() and rest.right()

    first, owner, fill = s[0], s[1], s[2:16]
    t0 = independent(load, owner, s[16:])
    t1 = independent(load, fill[0], [x for x in s[16:] if x is not t0])
    declined = pool.adr_held_workspace_declined()
    rest.run(first)                           # (alone in the pool: this use leaves no event)
    handed_on(owner, fill, t0)
    handed_on(fill[0], [first, t0, *fill[1:]], t1)
    assert pool.adr_held_workspace_declined() == declined


def test_an_outgrown_buffer_is_handed_on_in_order(pool):
    load, s = Load(), streams(8)
    owner = s[0]
    taker = independent(load, owner, s[1:])
    small, big, other = Product(pool, SMALL, 40), Product(pool, BIG, 41), Product(pool, SMALL, 42)
    load.put(owner)
    small.run(owner)
    done = mark(owner)
    big.run(owner)
    held = pool.adr_held_workspace_bytes()
    assert held > 2 * 16 * MIB                        # the old buffer and a larger one
    start = mark(taker)
    other.run(taker)
    end = mark(taker)
    running = not done.query()
    assert pool.adr_held_workspace_bytes() == held    # (the old one, not a new one)
    torch.cuda.synchronize()
    assert running and done.elapsed_time(start) < 0
    assert done.elapsed_time(end) > 0
    assert small.right() and big.right() and other.right()


def test_a_stream_s_buffer_serves_products_and_attention_in_turn(pool):
    s = torch.cuda.Stream()
    product = Product(pool, SMALL, 50)
    heads, n, d = 8, 3000, 128
    g = torch.Generator(device="cuda").manual_seed(51)
    q = torch.randn(heads, 1, d, dtype=torch.float16, device="cuda", generator=g)
    k, v = (torch.randn(heads, n, d, dtype=torch.float16, device="cuda", generator=g) for _ in range(2))
    outs = [torch.zeros(heads, 1, d, dtype=torch.float16, device="cuda") for _ in range(9)]

    def attention(out, stream):
        assert pool.adr_attention_f16(stream.cuda_stream, out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), heads,
                                      1, n, d, 1, d, d, 1, d, d, 1, d, n * d, 1, d, n * d, d ** -0.5, 1.0, 0) == 0
    attention(outs[8], s)
    torch.cuda.synchronize()
    assert pool.adr_held_workspace_bytes() == 16 * MIB  # it does take a buffer
    for i in range(8):
        product.run(s)
        attention(outs[i], s)
    assert pool.adr_held_workspace_bytes() == 16 * MIB
    torch.cuda.synchronize()
    assert product.right()
    assert all(torch.equal(o, outs[8]) for o in outs)
    scores = (q.double() * float(torch.tensor(d ** -0.5).half()) * k.double()).sum(-1, keepdim=True)
    want = (torch.softmax(scores, 1) * v.double()).sum(1, keepdim=True)
    # fp16 output and probabilities: 2^-11 of the largest value each, doubled
    assert ((outs[8].double() - want).abs().max() / want.abs().max()).item() <= 2e-3


@contextlib.contextmanager
def captured(stream):
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        graph.capture_begin()
        try:
            yield graph
        finally:
            graph.capture_end()


def replays(graph, a):
    for i in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert (a == 2 + i).all()


@pytest.mark.parametrize("alone", [True, False])
def test_release_on_a_stream_that_is_being_captured(pool, alone):
    """The buffer cannot be waited for then: the call says so, the buffer stays, and the capture goes on."""
    load, s = Load(), streams(2)
    product = Product(pool, SMALL, 60)
    a = torch.ones(256, dtype=torch.float16, device="cuda")
    if not alone:
        product.run(s[1])
    load.put(s[0])
    product.run(s[0])                                 # (alone in the pool this use leaves no event)
    before = pool.adr_held_workspace_bytes()
    with captured(s[0]) as graph:
        rc = pool.adr_release_held_workspace(s[0].cuda_stream)
        held = pool.adr_held_workspace_bytes()
        a.add_(1)
    assert rc > 0 and held == before
    replays(graph, a)
    assert product.right()
    assert pool.adr_release_held_workspace(s[0].cuda_stream) == 0
    assert pool.adr_held_workspace_bytes() == before - 16 * MIB


@pytest.mark.parametrize("alone", [True, False])
def test_release_while_another_stream_is_being_captured(pool, alone):
    load, s = Load(), streams(3)
    product = Product(pool, SMALL, 61)
    a = torch.ones(256, dtype=torch.float16, device="cuda")
    if not alone:
        product.run(s[2])
    load.put(s[0])
    product.run(s[0])
    done = mark(s[0])
    before = pool.adr_held_workspace_bytes()
    with captured(s[1]) as graph:
        rc = pool.adr_release_held_workspace(s[0].cuda_stream)
        held = pool.adr_held_workspace_bytes()
        a.add_(1)
    over = done.query()                               # (40 ms of work are not over by chance)
    assert rc == 0 and held == before - 16 * MIB and over
    assert product.right()
    replays(graph, a)
