"""Stacks of few angles, whose default batches are shallower and whose last slices
stay in the one launch: projections bit for bit the oracle's, adjoints bit for bit
those of another launch shape, on either side of the limits (12 and 24 angles, 400
pixels, 4e6 pixels times angles)."""
import numpy as np
import pytest

from trace_amd.phantom import angles_rad

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,P,S", [(30, 4, 9), (30, 13, 9), (260, 12, 20), (260, 13, 20),
                                   (60, 24, 31), (60, 25, 31), (400, 12, 33), (401, 12, 33),
                                   (260, 59, 40), (260, 60, 40)])
def test_default_shapes_at_few_angles(gpu, oracle, N, P, S):
    import torch
    from trace_amd import Projector
    th = angles_rad(P)
    center = N / 2.0 + 0.3
    rng = np.random.default_rng(N + P)
    x = rng.standard_normal((S, N, N)).astype(np.float32)
    r = torch.from_numpy(rng.standard_normal((P, S, N)).astype(np.float32)).cuda()
    with Projector(th, S, N, center, device=0) as pj:
        y = pj.forward(torch.from_numpy(x).cuda()).cpu().numpy()
        z = pj.adjoint(r)
    with Projector(th, S, N, center, device=0) as pj:
        pj.set_launch_shape(1, 32, 32, 8)
        other = pj.adjoint(r)
    assert torch.equal(z, other)
    want = oracle.forward(th, x, center)
    assert np.array_equal(y.view(np.int32), want.view(np.int32))


@pytest.mark.parametrize("alg", ["pml", "apmlr"])
@pytest.mark.parametrize("S", [33, 44])
def test_ordered_rest_in_its_own_launch(gpu, alg, S):
    """Enough angles for two launches: PML slice by slice; APMLR (whose slices are
    coupled) against the per-pixel form of the whole stack."""
    import torch
    from trace_amd import Projector
    N, P = 402, 26
    th = angles_rad(P)
    sino = np.random.default_rng(S).uniform(0.5, 2.0, (P, S, N)).astype(np.float32)

    def image(rows, tile):
        n = rows.shape[1]
        x = torch.ones((n, N, N), device="cuda:0")
        with Projector(th, n, N, N / 2.0 + 0.3, device=0) as pj:
            pj.set_ordered_tile(tile)
            pj.reconstruct(alg, 2, torch.from_numpy(np.ascontiguousarray(rows)).to("cuda:0"), x)
        return x.cpu().numpy()

    stack = image(sino, True)
    if alg == "apmlr":
        assert np.array_equal(stack.view(np.int32), image(sino, False).view(np.int32))
        return
    for s in sorted({0, 31, 32, S - 1}):
        alone = image(sino[:, s:s + 1], True)
        assert np.array_equal(stack[s].view(np.int32), alone[0].view(np.int32)), s
