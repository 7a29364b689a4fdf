"""Forward projections of images at the reach of 32-bit gathers: segments on the
far grid lines (indices past the image) add nothing.  The sums of a stack equal
those of its slices one by one, whose offsets are a half and an eighth as large."""
import numpy as np
import pytest

from trace_amd.phantom import angles_rad

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,S", [(23170, 2), (11585, 8)])
def test_stack_equals_its_slices(gpu, N, S):
    import torch
    from trace_amd import Projector
    th = angles_rad(1500)[:7]  # rays along the rows, the top grid line among them
    gen = torch.Generator(device="cuda").manual_seed(N)
    x = torch.rand((S, N, N), generator=gen, device="cuda")
    print(f"forward of {S} slices {N}^2", flush=True)
    with Projector(th, S, N, N / 2.0, device=0) as pj:
        pj.set_fwd_staged(False)
        assert pj.count_segments()[1] > 0  # segments outside the image
        y = pj.forward(x)
    with Projector(th, 1, N, N / 2.0, device=0) as pj:
        for s in range(S):
            one = pj.forward(x[s:s + 1])
            assert np.array_equal(y[:, s].cpu().numpy().view(np.int32),
                                  one[:, 0].cpu().numpy().view(np.int32)), s
