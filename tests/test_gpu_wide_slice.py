"""The largest image, 32768^2: one slice is past the reach of 32-bit gathers and
has a form of its own, in single calls and in a batch.  A few rays through it
against the oracle, and one iteration of a batch against the same call alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N, C = 32768, 24
THETA = np.float32([0.0, 0.4, 1.5707964, 2.2, 3.0])


def test_forward_of_the_largest_slice(gpu, oracle):
    import torch
    from trace_amd import Projector
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand((1, N, N), generator=gen, device="cuda")
    print(f"forward of one slice {N}^2", flush=True)
    with Projector(THETA, 1, C, C / 2.0 + 0.3, device=0, num_grids=N) as pj:
        y = pj.forward(x).cpu().numpy()
    want = oracle.forward(THETA, x.cpu().numpy(), C / 2.0 + 0.3, C=C)
    assert np.array_equal(y.view(np.int32), want.view(np.int32))


@pytest.mark.parametrize("alg", ["sirt", "mlem"])
def test_batched_largest_slice(gpu, alg):
    import torch
    from trace_amd import Projector
    from trace_amd.batch import Batch, BatchSlice
    gen = torch.Generator(device="cuda").manual_seed(2)
    sino = torch.rand((len(THETA), 1, C), generator=gen, device="cuda") + 0.5
    x0 = torch.rand((1, N, N), generator=gen, device="cuda") + 0.5
    print(f"batched {alg} of one slice {N}^2", flush=True)
    x = x0.clone()
    with Projector(THETA, 1, C, C / 2.0 + 0.3, device=0, num_grids=N) as pj:
        pj.reconstruct(alg, 1, sino, x)
    xb = x0[0].clone()
    sl = BatchSlice(THETA, sino[:, 0].contiguous(), xb, alg, 1, C / 2.0 + 0.3)
    with Batch([sl]) as b:
        b.run()
    torch.cuda.synchronize()
    # bits: pixels without a ray hold 0 / 0
    assert torch.equal(x[0].view(torch.int32), xb.view(torch.int32))
    crossed = torch.isfinite(xb)
    assert crossed.any() and (xb != x0[0])[crossed].any()
