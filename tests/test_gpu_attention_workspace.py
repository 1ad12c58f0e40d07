"""adr_attention_f16_ws: keys shared through the caller's buffer in every context alike, and with no buffer
one launch that allocates nothing and gives the same bits eagerly and under capture.  Reference: the
same attention in float64."""
import pytest
import torch

from adrastea_amd import GpuKernels, MatmulMask, TensorView, _ffi
from adrastea_amd import kernels as K

pytestmark = pytest.mark.gpu

# fp16 output and probabilities: 2^-11 of the largest value each, doubled
TOL = 2e-3


class Attention:
    def __init__(self, heads, m, n, d, causal, seed=1):
        g = torch.Generator(device="cuda").manual_seed(seed)
        self.q, self.k, self.v = (torch.randn(heads, r, d, device="cuda", dtype=torch.float16, generator=g) for r in (m, n, n))
        self.out = torch.zeros_like(self.q)
        self.scale, self.mask = d ** -0.5, MatmulMask.CAUSAL if causal else MatmulMask.NONE
        self.views = [TensorView.of(t) for t in (self.out, self.q, self.k, self.v)]
        s = self.q.double() @ self.k.double().transpose(1, 2).contiguous() * float(torch.tensor(self.scale).half())
        if causal:
            s = s.masked_fill(torch.arange(n, device="cuda")[None] > torch.arange(m, device="cuda")[:, None], float("-inf"))
        self.want = torch.softmax(s, -1) @ self.v.double()
        self.need = K.attention_workspace_bytes(*[x.layout for x in self.views], self.mask)

    def run(self, workspace, nbytes):
        heads, m, d = self.q.shape
        strides = [s for x in self.views for s in (1, d, x.layout.strides[0])]
        self.out.fill_(7)
        rc = _ffi.lib().adr_attention_f16_ws(torch.cuda.current_stream().cuda_stream,
                                             *[x.data_ptr() for x in self.views], heads, m, self.k.shape[1], d, *strides,
                                             self.scale, 1.0, self.mask, workspace, nbytes)
        assert rc == 0, _ffi.strerror(rc)

    def result(self):
        torch.cuda.synchronize()
        assert ((self.out.double() - self.want).abs().max() / self.want.abs().max()).item() <= TOL
        return self.out.clone()


SHAPES = [(32, 1, 2047, 128, False), (3, 16, 3001, 64, False), (1, 40, 2000, 128, False), (2, 900, 900, 64, True)]


@pytest.mark.parametrize("shape", SHAPES)
def test_the_same_bits_eagerly_and_under_capture(shape):
    a = Attention(*shape)
    assert a.need > 0
    guard = torch.full((a.need + 64,), 0x5a, dtype=torch.uint8, device="cuda")
    results = {}
    for name, ptr, nbytes in (("all", guard.data_ptr(), a.need), ("less", guard.data_ptr(), a.need - 1), ("none", None, 0)):
        K.set_held_workspace_limit(_ffi.HELD_WORKSPACE_DEFAULT_BYTES)   # (the pool is never touched)
        K.release_held_workspace("all")
        a.run(ptr, nbytes)
        eager = a.result()
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph):
            a.run(ptr, nbytes)
        for _ in range(3):
            a.out.zero_()
            graph.replay()
            assert torch.equal(a.result(), eager)
            a.q.mul_(1.0)   # (eager work between the replays)
        assert K.held_workspace_bytes() == 0
        results[name] = eager
    assert (guard[a.need:] == 0x5a).all()
    K.set_held_workspace_limit(0)                                       # the pool off: as with no buffer
    GpuKernels().attention_f16(*a.views, a.scale, 1.0, a.mask)
    assert torch.equal(a.result(), results["none"])
    K.set_held_workspace_limit(_ffi.HELD_WORKSPACE_DEFAULT_BYTES)       # through the pool: as with all of it
    GpuKernels().attention_f16(*a.views, a.scale, 1.0, a.mask)
    assert K.held_workspace_bytes() > 0
    assert torch.equal(a.result(), results["all"])
    K.release_held_workspace("all")
    GpuKernels(workspace_bytes=a.need).attention_f16(*a.views, a.scale, 1.0, a.mask)
    assert torch.equal(a.result(), results["all"])
    assert K.held_workspace_bytes() == 0
