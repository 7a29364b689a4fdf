"""The forward projector with several lanes per ray: bit-identical to the
oracle's sums in the reference's order, at piece boundaries (rays of 16 segments
and around, and of K * 16), with columns outside the image, off-centre axes,
axis-aligned rays on grid lines, and angles whose lists cannot be entered in the
middle (below -pi/2)."""
import numpy as np
import pytest

from trace_amd.phantom import angles_rad

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [1, 2, 4, 7, 20])
@pytest.mark.parametrize("N,C,P,offset", [(8, 8, 5, 0.0), (16, 19, 7, 0.5), (33, 33, 9, -1.3),
                                          (64, 50, 6, 2.0), (129, 129, 8, 0.5)])
def test_forward_split_bitexact(gpu, oracle, S, N, C, P, offset):
    import torch
    from trace_amd import Projector
    th = np.concatenate([angles_rad(P), np.float32([-0.4, -2.1, -3.0, 3.7, 5.5])])
    x = np.random.default_rng(N + S).standard_normal((S, N, N)).astype(np.float32)
    ctr = C / 2.0 + offset
    with Projector(th, S, C, ctr, device=0, num_grids=N) as pj:
        y = pj.forward(torch.from_numpy(x).to("cuda:0")).cpu().numpy()
    want = oracle.forward(th, x, ctr, C=C)
    assert np.array_equal(y.view(np.int32), want.view(np.int32))


@pytest.mark.parametrize("alg", ["sirt", "mlem"])
@pytest.mark.parametrize("S", [1, 2, 4])
def test_weights_split_as_in_a_stack(gpu, alg, S):
    """The ray weights and their maxima: slices reconstructed with several
    lanes per ray equal the same slices of a 33-slice stack."""
    import torch
    from trace_amd import Projector
    N, P = 70, 60
    th = angles_rad(P)
    sino = np.random.default_rng(3).uniform(0.5, 2.0, (P, 33, N)).astype(np.float32)
    out = []
    for n in (33, S):
        x = torch.full((n, N, N), 0.0 if alg == "sirt" else 1.0, device="cuda:0")
        with Projector(th, n, N, N / 2.0 + 0.7, device=0) as pj:
            pj.reconstruct(alg, 3, torch.from_numpy(sino[:, :n].copy()).to("cuda:0"), x)
        out.append(x.cpu().numpy())
    assert np.array_equal(out[0][:S].view(np.int32), out[1].view(np.int32))
