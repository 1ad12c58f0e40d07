"""GPU parity of adr_attention_f16 at the edges of its kernels: the tiles of 64 keys and 128 query rows,
the two groups of wavefronts that share a workgroup's keys, the parts that several workgroups leave
in a workspace (and the same shapes without one), the kernel of at most sixteen query rows, and rows
closer together than they are long.  Reference: the same attention in float64 on the CPU."""
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


def test_more_workgroups_than_fit():
    run(40, 1700, 1700, 128, True)   # 560 blocks: dealt out from the longest to the shortest
    run(32, 1100, 300, 64, False)


@pytest.mark.parametrize("m,causal", [(1, False), (33, False), (130, True)])
def test_keys_that_overlap(m, causal):
    """A window over a signal: key rows of 64 elements, 8 apart (rows closer than they are long)."""
    n, d = 300, 64
    g = torch.Generator(device="cuda").manual_seed(3)
    signal = torch.randn(n * 8 + d, device="cuda", dtype=torch.float16, generator=g)
    v = torch.randn(n, d, device="cuda", dtype=torch.float16, generator=g)
    q = torch.randn(m, d, device="cuda", dtype=torch.float16, generator=g)
    out = torch.zeros(m, d, device="cuda", dtype=torch.float16)
    keys = TensorView(signal, TensorLayout((n, d), (8, 1)))
    GpuKernels().attention_f16(TensorView.of(out), TensorView.of(q), keys, TensorView.of(v), d ** -0.5, 1.0,
                               MatmulMask.CAUSAL if causal else MatmulMask.NONE)
    k = signal.as_strided((n, d), (8, 1))
    want = reference(q[None], k[None], v[None], d ** -0.5, causal)[0]
    assert ((out.double().cpu() - want).abs().max() / want.abs().max()).item() <= TOL


def test_under_capture_no_buffer_is_used():
    heads, n, d = 8, 3000, 128
    g = torch.Generator(device="cuda").manual_seed(4)
    q, k, v = (torch.randn(heads, r, d, device="cuda", dtype=torch.float16, generator=g) for r in (1, n, n))
    out = torch.zeros(heads, 1, d, device="cuda", dtype=torch.float16)
    kern = GpuKernels()
    K.release_held_workspace("all")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        kern.attention_f16(TensorView.of(out), TensorView.of(q), TensorView.of(k), TensorView.of(v), d ** -0.5)
    assert K.held_workspace_bytes() == 0
    want = reference(q, k, v, d ** -0.5, False)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert ((out.double().cpu() - want).abs().max() / want.abs().max()).item() <= TOL
        q.mul_(1.0)  # (eager work between the replays)
