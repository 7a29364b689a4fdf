"""Column sums of the largest image with rays on its right edge line (wrapped
segments): the tile form for such rays would be a launch of 2^32 lanes there, so
the per-pixel form serves.  Bit for bit the sums of the oracle's segments in
order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [32760, 32768])
def test_edge_rays_of_the_largest_image(gpu, oracle, N):
    from trace_amd import Projector
    C, th = 24, np.float32([1.5707964, 0.0])
    center = C / 2 + N / 2 + 0.5  # column 12 of the first projection lies on x = N/2
    rays = oracle.trace_rays(N, C, center, np.repeat(th, C), np.tile(np.arange(C), 2))
    _, idx, ln = rays
    assert np.count_nonzero(idx % N == 0) > 1000  # wrapped onto column 0
    ok = (idx >= 0) & (idx < N * N)
    idx, ln = idx[ok], ln[ok]
    touched, where = np.unique(idx, return_inverse=True)
    want = np.zeros(touched.size, np.float32)
    np.add.at(want, where, ln)  # one after the other
    print(f"column sums {N}^2 with rays on the edge line", flush=True)
    with Projector(th, 1, C, center, device=0, num_grids=N) as pj:
        den = pj.column_sums().reshape(-1).cpu().numpy()
    assert np.array_equal(den[touched].view(np.int32), want.view(np.int32))
    assert np.count_nonzero(den) == np.count_nonzero(want)
