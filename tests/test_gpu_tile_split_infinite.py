"""Shared tiles with an infinite weight: the batch is summed by one workgroup a
tile.  Its finite slices keep their integer sums (bit for bit those of tiles that
are not shared); the slice with the infinity is summed in float, within the
rounding of its own terms of the float64 sum, and not finite exactly in the
pixels that the ray with the infinite weight crosses."""
import numpy as np
import pytest

from trace_amd.phantom import angles_rad

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [1, 2, 4, 8])
@pytest.mark.parametrize("p,c", [(17, 20), (0, 0), (299, 39)])
def test_infinite_weight_in_shared_tiles(gpu, oracle, S, p, c):
    import torch
    from trace_amd import Projector
    N, P = 40, 300
    center = N / 2.0 + 0.3
    th = angles_rad(P)
    r = np.random.default_rng(S).standard_normal((P, S, N)).astype(np.float32)
    r[p, S - 1, c] = np.inf
    d = torch.from_numpy(r).to("cuda:0")
    z = []
    for side in (16, 32):
        with Projector(th, S, N, center, device=0) as pj:
            pj.set_launch_shape(1, side, side, S)
            z.append(pj.adjoint(d).cpu().numpy())
            counts = pj.segment_counts().cpu().numpy()
    assert np.array_equal(z[0][:S - 1].view(np.int32), z[1][:S - 1].view(np.int32))

    idx, ln, _ = oracle.trace_ray(N, N, center, th[p], c)
    crossed = np.zeros(N * N, bool)
    crossed[idx[(idx >= 0) & (idx < N * N)]] = True
    crossed = crossed.reshape(N, N)
    assert crossed.any()
    rest = r[:, S - 1:].copy()
    rest[p, 0, c] = 0.0
    want = oracle.adjoint(th, rest, center)[0]
    size = oracle.adjoint(th, np.abs(rest), center)[0]
    # n products and sums in float, each within 2^-24 of the sum of magnitudes
    bound = (counts + 1) * 2.0 ** -24 * size
    for v in (z[0][S - 1], z[1][S - 1]):
        assert np.array_equal(~np.isfinite(v), crossed)
        assert (np.abs(v - want)[~crossed] <= bound[~crossed]).all()
