"""Projections and adjoints captured into a HIP graph after another call has
prepared the handle: a capture can neither allocate nor copy tables up, so what
such a call finds missing must not be needed.  Each graph is replayed several
times, on new inputs, with eager calls and synchronisation between."""
import numpy as np
import pytest

from trace_amd.phantom import angles_rad

pytestmark = pytest.mark.gpu


def _replay(torch, stream, call, reference, src, dst, inputs):
    graph = torch.cuda.CUDAGraph()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=stream):
        call(src, dst)
    for v in inputs:
        src.copy_(v)
        dst.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        want = reference(v)
        torch.cuda.synchronize()
        assert np.array_equal(dst.cpu().numpy().view(np.int32), want.cpu().numpy().view(np.int32))


@pytest.mark.parametrize("warm", ["sirt", "pml"])
@pytest.mark.parametrize("N,P,S", [(64, 300, 1), (64, 300, 3), (260, 40, 1), (96, 60, 7)])
def test_adjoint_after_a_reconstruction(gpu, N, P, S, warm):
    """Small images share a tile's angles among workgroups, which takes a
    workspace that a regularised reconstruction and segment counts do not; and
    one slice is reconstructed without the slice-batched copy."""
    import torch
    from trace_amd import Projector
    th = angles_rad(P)
    s = torch.cuda.Stream()
    gen = torch.Generator(device="cuda").manual_seed(N + S)
    r = [torch.rand((P, S, N), generator=gen, device="cuda") - 0.3 for _ in range(3)]
    z = torch.empty((S, N, N), device="cuda")
    print(f"captured adjoint N={N} P={P} S={S} after {warm}", flush=True)
    with Projector(th, S, N, N / 2.0 + 0.3, device=0, stream=s.cuda_stream) as pj, \
            Projector(th, S, N, N / 2.0 + 0.3, device=0) as eager:
        with torch.cuda.stream(s):
            pj.reconstruct(warm, 1, r[0].abs() + 0.1, torch.ones_like(z))
            if warm == "pml":  # whose sums need no column counts
                pj.segment_counts()
        torch.cuda.synchronize()
        _replay(torch, s, lambda a, b: pj.adjoint(a, out=b), lambda v: eager.adjoint(v),
                torch.empty_like(r[0]), z, r)


@pytest.mark.parametrize("N,P,S", [(64, 300, 1), (96, 60, 3), (96, 60, 12), (64, 48, 32)])
def test_forward_after_an_adjoint(gpu, N, P, S):
    """The slab-staged form's plan is made by the first projection; captured,
    that one takes another form with the same sums."""
    import torch
    from trace_amd import Projector
    th = angles_rad(P)
    s = torch.cuda.Stream()
    gen = torch.Generator(device="cuda").manual_seed(N + S)
    x = [torch.rand((S, N, N), generator=gen, device="cuda") for _ in range(3)]
    y = torch.empty((P, S, N), device="cuda")
    print(f"captured forward N={N} P={P} S={S}", flush=True)
    with Projector(th, S, N, N / 2.0 + 0.3, device=0, stream=s.cuda_stream) as pj, \
            Projector(th, S, N, N / 2.0 + 0.3, device=0) as eager:
        pj.set_fwd_staged(True)
        eager.set_fwd_staged(False)
        with torch.cuda.stream(s):
            pj.adjoint(torch.ones_like(y))
        torch.cuda.synchronize()
        _replay(torch, s, lambda a, b: pj.forward(a, out=b), lambda v: eager.forward(v),
                torch.empty_like(x[0]), y, x)
        # afterwards, out of a capture, the plan is made
        with torch.cuda.stream(s):
            again = pj.forward(x[0])
        torch.cuda.synchronize()
        assert torch.equal(again, eager.forward(x[0]))
