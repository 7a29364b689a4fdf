"""Tiles whose angles are shared among workgroups: integer sums, so the
backprojection equals that of tiles of another size, which are not shared, bit
for bit.  Image sides around the tile's, uneven shares of the angles, axis-aligned
rays on grid lines, a slice with infinite weights (summed in float by one
workgroup), and launches one after the other on one handle (the counters that
tell the last workgroup)."""
import numpy as np
import pytest

from trace_amd.phantom import angles_rad

pytestmark = pytest.mark.gpu

SHAPES = {1: (1, 1), 2: (2, 2), 4: (4, 4), 7: (8, 8), 16: (16, 16), 33: (32, 16)}


@pytest.mark.parametrize("S", sorted(SHAPES))
@pytest.mark.parametrize("N,P,offset", [(5, 331, 0.0), (16, 400, 0.5), (17, 257, 1.3),
                                        (63, 500, 0.5), (81, 336, -3.0), (125, 190, 1.5)])
def test_split_equals_unsplit(gpu, S, N, P, offset):
    import torch
    from trace_amd import Projector
    th = angles_rad(P)
    r = np.random.default_rng(N * S).standard_normal((2, P, S, N)).astype(np.float32)
    r = torch.from_numpy(r).to("cuda:0")
    sb, other = SHAPES[S]
    z = []
    for shape in ((16, 16, sb), (32, 32, other)):
        with Projector(th, S, N, N / 2.0 + offset, device=0) as pj:
            pj.set_launch_shape(1, *shape)
            z.append([pj.adjoint(v).cpu().numpy() for v in (r[0], r[1], r[0])])
    for a, b in zip(*z):
        assert np.array_equal(a.view(np.int32), b.view(np.int32))


@pytest.mark.parametrize("S", [1, 4])
def test_split_with_infinite_weights(gpu, S):
    import torch
    from trace_amd import Projector
    N, P = 40, 300
    th = angles_rad(P)
    r = np.random.default_rng(1).standard_normal((P, S, N)).astype(np.float32)
    r[17, S - 1, 20] = np.inf
    r = torch.from_numpy(r).to("cuda:0")
    z = []
    for side in (16, 32):
        with Projector(th, S, N, N / 2.0, device=0) as pj:
            pj.set_launch_shape(1, side, side, S)
            z.append(pj.adjoint(r).cpu().numpy())
    fin = np.isfinite(z[0])
    assert np.array_equal(fin, np.isfinite(z[1])) and not fin[S - 1].all()
    # float sums in any order: n terms of at most max |r| sqrt 2 each
    bound = 2.0 * 6 * P * 2.0 ** -24 * 6 * P * np.sqrt(2) * 6
    assert np.abs(z[0][fin] - z[1][fin]).max() <= bound
