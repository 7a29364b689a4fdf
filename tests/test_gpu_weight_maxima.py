"""Per-slice largest weights, which set the fixed-point scale of the tile
backprojector: a slice of a stack must come out as it does alone, bit for bit,
whatever the magnitude of the slices beside it (the transposition in blocks of
64 columns x 32 slices and the maxima it raises; one slice is read in place)."""
import numpy as np
import pytest

from trace_amd.phantom import angles_rad

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,N,P", [(1, 64, 5), (2, 65, 7), (5, 63, 9), (32, 40, 6), (33, 70, 4),
                                   (70, 48, 3)])
def test_adjoint_slices_alone(gpu, S, N, P):
    import torch
    from trace_amd import Projector
    th = angles_rad(P)
    rng = np.random.default_rng(S * 100 + N)
    r = rng.standard_normal((P, S, N)).astype(np.float32)
    r *= np.ldexp(1.0, rng.integers(-20, 20, S)).astype(np.float32)[None, :, None]
    d = torch.from_numpy(r).to("cuda:0")
    with Projector(th, S, N, N / 2.0, device=0) as pj:
        z = pj.adjoint(d).cpu().numpy()
    with Projector(th, 1, N, N / 2.0, device=0) as one:
        for s in range(S):
            z1 = one.adjoint(d[:, s:s + 1].contiguous()).cpu().numpy()
            assert np.array_equal(z[s].view(np.int32), z1[0].view(np.int32)), s
