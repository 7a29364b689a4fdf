"""Stacks whose last 32-slice batch would be mostly empty: the backprojectors
take the rest in a second launch with a batch of its own.  Every slice must come
out as with one launch (an explicit launch shape), and as it does alone."""
import numpy as np
import pytest

from trace_amd.phantom import angles_rad

pytestmark = pytest.mark.gpu

P = 9


@pytest.mark.parametrize("S", [32, 33, 35, 41, 48, 49, 66])
def test_adjoint_in_two_launches(gpu, S):
    N = 260
    import torch
    from trace_amd import Projector
    th = angles_rad(P)
    r = np.random.default_rng(S).standard_normal((P, S, N)).astype(np.float32)
    r *= np.ldexp(1.0, np.arange(S) % 23 - 11).astype(np.float32)[None, :, None]
    d = torch.from_numpy(r).to("cuda:0")
    z = []
    for one in (False, True):
        with Projector(th, S, N, N / 2.0 + 0.3, device=0) as pj:
            if one:
                pj.set_launch_shape(32, 16, 16, 32)
            z.append(pj.adjoint(d).cpu().numpy())
    assert np.array_equal(z[0].view(np.int32), z[1].view(np.int32))


@pytest.mark.parametrize("alg", ["pml", "apmlr"])
@pytest.mark.parametrize("S", [33, 44, 66])
def test_ordered_in_two_launches(gpu, alg, S):
    """PML slice by slice; APMLR against the per-pixel form of the whole stack
    (its slices are coupled)."""
    import torch
    from trace_amd import Projector
    N = 402
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
