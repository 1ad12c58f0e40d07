"""GPU parity of adr_attention_f16 at the edges of its kernels: the tiles of 64 keys and 128 query rows,
the two groups of wavefronts that share a workgroup's keys, the parts that several workgroups leave
in a workspace (and the same shapes without one), the kernel of at most sixteen query rows, and rows
closer together than they are long or further apart than 32-bit offsets reach.  Reference: the same
attention in float64 on the CPU."""
import contextlib

import pytest
import torch

from adrastea_amd import GpuKernels, MatmulMask, TensorLayout, TensorView, _ffi
from adrastea_amd import kernels as K

pytestmark = pytest.mark.gpu

# fp16 output (half a step of the largest value is 2^-11 of it) and probabilities rounded to fp16
# (2^-11 of each term, and the terms' magnitudes sum to at most the largest value): 2^-10, doubled
TOL = 2e-3


def reference(q, k, v, scale, causal):
    """[heads, m, d], [heads, n, d] -> [heads, m, d] in float64; the scale rounded to fp16 as the matmul's."""
    q, k, v = (t.double().cpu() for t in (q, k, v))
    s = q @ k.transpose(1, 2) * float(torch.tensor(scale).half())
    if causal:
        m, n = s.shape[-2:]
        s = s.masked_fill(torch.arange(n)[None, :] > torch.arange(m)[:, None], float("-inf"))
    return torch.softmax(s, -1) @ v


def run(heads, m, n, d, causal, seed=1):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = (torch.randn(r, heads * d, device="cuda", dtype=torch.float16, generator=g) for r in (m, n, n))
    # rows before and after the output show what is written outside it
    guard = torch.full((m + 2, heads * d), 7.0, dtype=torch.float16, device="cuda")
    out = guard[1:m + 1]

    def view(t):
        return TensorView.of(t).shape_cast([t.shape[0], heads, d]).permute([1, 0, 2])
    GpuKernels().attention_f16(view(out), view(q), view(k), view(v), d ** -0.5, 1.0,
                               MatmulMask.CAUSAL if causal else MatmulMask.NONE)
    assert (guard[0] == 7).all() and (guard[-1] == 7).all()

    def heads_of(t):
        return t.view(t.shape[0], heads, d).permute(1, 0, 2)
    want = reference(heads_of(q), heads_of(k), heads_of(v), d ** -0.5, causal)
    got = heads_of(out).double().cpu()
    assert torch.isfinite(got).all()
    err = ((got - want).abs().max() / want.abs().max()).item()
    assert err <= TOL, err
    return out.clone()


@contextlib.contextmanager
def pool_on():
    limit = K.held_workspace_limit()
    try:
        K.set_held_workspace_limit(_ffi.HELD_WORKSPACE_DEFAULT_BYTES)
        K.release_held_workspace("all")
        yield
    finally:
        K.set_held_workspace_limit(limit)
        K.release_held_workspace("all")


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n", [1, 15, 31, 32, 33, 63, 64, 65, 127, 129, 191, 193, 257])
def test_key_tiles(d, n):
    for m in (1, 16, 17, 40):
        run(2, m, n, d, False)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("m", [17, 31, 32, 33, 127, 128, 129, 255, 257])
def test_query_blocks(d, m):
    run(3, m, 70, d, False)
    run(3, m, m, d, True)
    run(2, m, 40, d, True)       # fewer keys than rows: the last rows see all of them
    run(2, m, m + 100, d, True)  # more: the last keys are seen by none


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n", [320, 321, 384, 385, 449, 512, 575, 640, 703])
def test_two_groups_of_wavefronts(d, n):
    """Tiles that divide evenly between the groups and that do not, group 1 without work under the mask."""
    run(2, n, n, d, True)
    run(2, 130, n, d, False)


@pytest.mark.parametrize("heads,m,n,d", [(29, 1025, 1025, 128), (33, 1024, 1024, 64), (26, 1410, 1410, 64), (32, 1100, 1030, 64),
                                         (40, 1101, 1300, 128)])
def test_two_groups_of_wavefronts_in_a_second_round(heads, m, n, d):
    """Under the mask with up to half as many query blocks again as compute units (261 ... 384 of 256 here), from
    1024 keys that some row sees on; heads that do and do not divide by the dies, and a few rows past a block."""
    run(heads, m, n, d, True)


@pytest.mark.parametrize("heads,m,n,d", [(4, 1, 2048, 128), (4, 1, 2047, 128), (3, 16, 3001, 64), (5, 9, 4100, 64),
                                         (1, 40, 2000, 128), (2, 130, 1500, 64), (1, 17, 8192, 128)])
def test_keys_shared_by_workgroups(heads, m, n, d):
    limit = K.held_workspace_limit()
    try:
        K.set_held_workspace_limit(_ffi.HELD_WORKSPACE_DEFAULT_BYTES)
        K.release_held_workspace("all")
        shared = run(heads, m, n, d, False)
        assert K.held_workspace_bytes() > 0   # (the parts went through a buffer of the pool)
        again = run(heads, m, n, d, False)
        assert torch.equal(shared, again)     # parts are added in a fixed order
        K.set_held_workspace_limit(0)         # no buffer: every block walks all keys
        run(heads, m, n, d, False)
    finally:
        K.set_held_workspace_limit(limit)
        K.release_held_workspace("all")


@pytest.mark.parametrize("heads,m,n,d", [(2, 900, 900, 64), (1, 700, 700, 64), (1, 700, 600, 128), (1, 600, 600, 64),
                                         (2, 700, 2000, 64), (1, 1000, 600, 64)])
def test_keys_shared_by_workgroups_under_the_mask(heads, m, n, d):
    """A query block's tiles end at the diagonal: parts of unequal length, and parts of the first blocks
    without any tile, whose sums of nothing must not count."""
    with pool_on():
        shared = run(heads, m, n, d, True)
        assert K.held_workspace_bytes() > 0
        assert torch.equal(shared, run(heads, m, n, d, True))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("m", [17, 31, 33, 64, 65, 79, 80, 81])
def test_one_tile_of_keys(m, d):
    for n in (1, 5, 31, 33, 63, 64, 65):
        run(3, m, n, d, False)
        run(3, m, n, d, True)
    run(2, min(m, 64), 200, d, True)   # more keys, but only a tile of them is seen
    run(2, 7, 64, d, True)


def test_more_workgroups_than_fit():
    run(40, 1700, 1700, 128, True)   # 560 blocks: dealt out from the longest to the shortest
    run(32, 1100, 300, 64, False)


@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("m,causal", [(1, False), (33, False), (500, True)])
def test_keys_that_overlap(m, causal, shared):
    """A window over a signal: key rows of 64 elements, 8 apart (rows closer than they are long)."""
    n, d = 600, 64
    g = torch.Generator(device="cuda").manual_seed(3)
    signal = torch.randn(n * 8 + d, device="cuda", dtype=torch.float16, generator=g)
    v = torch.randn(n, d, device="cuda", dtype=torch.float16, generator=g)
    q = torch.randn(m, d, device="cuda", dtype=torch.float16, generator=g)
    out = torch.zeros(m, d, device="cuda", dtype=torch.float16)
    keys = TensorView(signal, TensorLayout((n, d), (8, 1)))
    with pool_on() if shared else contextlib.nullcontext():
        GpuKernels().attention_f16(TensorView.of(out), TensorView.of(q), keys, TensorView.of(v), d ** -0.5, 1.0,
                                   MatmulMask.CAUSAL if causal else MatmulMask.NONE)
        assert (K.held_workspace_bytes() > 0) == shared
    k = signal.as_strided((n, d), (8, 1))
    want = reference(q[None], k[None], v[None], d ** -0.5, causal)[0]
    assert ((out.double().cpu() - want).abs().max() / want.abs().max()).item() <= TOL


# (query rows, keys, elements between query rows, between key and value rows)
FAR = [(40, 50, 1 << 22, 1 << 25),             # one tile; a head of 2^30 elements and more
       (40, 70, 1 << 22, 1 << 22),             # rows of 8 MiB: two tiles do not fit the offsets
       (40, 600, 1 << 21, 1 << 21),            # a head of 2^30 elements and more
       (3, 70, 512, 1 << 22),
       (257, 600, 1 << 22, 512)]               # query rows alone


@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("m,n,far_q,far_k", FAR)
def test_rows_far_apart(m, n, far_q, far_k, d, shared):
    heads = 2
    assert max(m * far_q, n * far_k) >= 1 << 30 or far_k >= 1 << 22
    g = torch.Generator(device="cuda").manual_seed(7)

    def far_rows(rows, far, columns):
        t = torch.empty((rows - 1) * far + columns, dtype=torch.float16, device="cuda")
        view = t.as_strided((rows, columns), (far, 1))
        view.copy_(torch.randn(rows, columns, dtype=torch.float16, device="cuda", generator=g))
        return t, view

    def heads_view(t, rows, far, offset=0):
        return TensorView(t, TensorLayout((heads, rows, d), (d, far, 1)), offset)
    (qt, q), (kvt, kv) = far_rows(m, far_q, heads * d), far_rows(n, far_k, 2 * heads * d)
    k, v = kv[:, :heads * d], kv[:, heads * d:]
    for causal in (False, True):
        out = torch.full((m, heads * d), 7.0, dtype=torch.float16, device="cuda")
        with pool_on() if shared else contextlib.nullcontext():
            GpuKernels().attention_f16(heads_view(out, m, heads * d), heads_view(qt, m, far_q), heads_view(kvt, n, far_k),
                                       heads_view(kvt, n, far_k, heads * d), d ** -0.5, 1.0,
                                       MatmulMask.CAUSAL if causal else MatmulMask.NONE)
        q3, k3, v3 = (t.reshape(-1, heads, d).permute(1, 0, 2) for t in (q, k, v))
        want = reference(q3, k3, v3, d ** -0.5, causal)
        got = out.view(m, heads, d).permute(1, 0, 2).double().cpu()
        assert ((got - want).abs().max() / want.abs().max()).item() <= TOL


@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("heads,m,n,d", [(4, 3, 2048, 128),   # at most sixteen rows, its four wavefronts; parts
                                         (3, 16, 1000, 64),
                                         (2, 40, 64, 128),    # one tile
                                         (2, 40, 300, 64),    # one group
                                         (2, 130, 640, 64),   # two groups; parts
                                         (2, 40, 2000, 128)])
def test_infinities_and_nan_pass_through_the_merges(heads, m, n, d, shared):
    """Wavefronts, groups and workgroups that share keys add up results of which some have seen no key that
    counts (every score of theirs -inf), and some an infinity or a NaN: as the sum over all keys would."""
    g = torch.Generator(device="cuda").manual_seed(8)
    q, k, v = (torch.randn(heads, r, d, device="cuda", dtype=torch.float16, generator=g) for r in (m, n, n))
    q[..., 0] = 1.0
    tile32, tile64 = torch.arange(n, device="cuda") // 32, torch.arange(n, device="cuda") // 64
    masked = {"none": tile32 < 0, "first half": tile64 < n // 128, "second half": tile64 >= n // 128,
              "even tiles": tile64 % 2 == 0, "odd tiles": tile64 % 2 == 1, "one wavefront's": tile32 % 4 != 1,
              "all but the last key": torch.arange(n, device="cuda") != n - 1, "all": tile32 >= 0}

    def check(what, k, v):
        out = torch.zeros(heads, m, d, device="cuda", dtype=torch.float16)
        with pool_on() if shared else contextlib.nullcontext():
            GpuKernels().attention_f16(*(TensorView.of(t) for t in (out, q, k, v)), d ** -0.5)
        want, got = reference(q, k, v, d ** -0.5, False), out.double().cpu()
        assert torch.equal(got.isnan(), want.isnan()), what
        whole = want.isfinite()
        assert torch.equal(got.isfinite(), whole), what
        infinite = want.isinf()
        assert torch.equal(got[infinite], want[infinite]), what
        if whole.any():
            assert ((got - want)[whole].abs().max() / want[whole].abs().max()).item() <= TOL, what

    inf, nan = float("inf"), float("nan")
    for what, keys in masked.items():
        x = k.clone()
        x[:, keys, 0] = -inf
        check(what + " masked by -inf", x, v)
    for key in (0, n // 2, n - 1):
        for value in (inf, nan):
            x = k.clone()
            x[0, key, 0] = value
            check(f"key {key} {value}", x, v)
            x = v.clone()
            x[0, key, 5] = value
            x[-1, key, d - 1] = -value
            check(f"value {key} {value}", k, x)


def test_under_capture_no_buffer_is_used():
    heads, n, d = 8, 3000, 128
    g = torch.Generator(device="cuda").manual_seed(4)
    q, k, v = (torch.randn(heads, r, d, device="cuda", dtype=torch.float16, generator=g) for r in (1, n, n))
    out = torch.zeros(heads, 1, d, device="cuda", dtype=torch.float16)
    kern = GpuKernels()

    def call():
        kern.attention_f16(TensorView.of(out), TensorView.of(q), TensorView.of(k), TensorView.of(v), d ** -0.5)
    with pool_on():
        call()
        torch.cuda.synchronize()
        assert K.held_workspace_bytes() > 0   # eagerly the call does take one
        K.release_held_workspace("all")
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            call()
        assert K.held_workspace_bytes() == 0
    call()                                    # (the pool is off again: as under capture)
    torch.cuda.synchronize()
    unshared = out.clone()
    want = reference(q, k, v, d ** -0.5, False)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, unshared)
        assert ((out.double().cpu() - want).abs().max() / want.abs().max()).item() <= TOL
        q.mul_(1.0)  # (eager work between the replays)
