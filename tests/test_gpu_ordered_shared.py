"""The ordered sums with several wavefronts per tile against the per-pixel form:
the same float sums bit for bit, for tile counts on either side of the choices
(8, 4 wavefronts and 1), stacks that do not fill their batch, and geometries with
wrapped segments (rays on the right edge line: whole or half pixel shifts)."""
import numpy as np
import pytest

from trace_amd.phantom import angles_rad

pytestmark = pytest.mark.gpu

CASES = [  # N, P, S, axis offset
    (24, 45, 1, 0.0), (24, 45, 3, 0.5), (64, 50, 5, 0.5), (81, 37, 20, 0.3), (81, 37, 33, 2.5),
    (88, 30, 9, -1.5), (96, 30, 2, 0.0), (129, 40, 11, 0.5), (200, 24, 18, -3.0), (330, 12, 6, 1.5)]


@pytest.mark.parametrize("alg", ["pml", "apmlr", "sirt"])
@pytest.mark.parametrize("N,P,S,offset", CASES)
def test_shared_equals_per_pixel(gpu, alg, N, P, S, offset):
    import torch
    from trace_amd import Projector
    th = angles_rad(P)
    rng = np.random.default_rng(N + S)
    sino = torch.from_numpy(rng.uniform(0.5, 2.0, (P, S, N)).astype(np.float32)).to("cuda:0")
    out, den = [], []
    for tile in (True, False):
        x = torch.full((S, N, N), 0.0 if alg == "sirt" else 1.0, device="cuda:0")
        with Projector(th, S, N, N / 2.0 + offset, device=0) as pj:
            pj.set_ordered_tile(tile)
            if alg == "sirt":
                pj.set_ordered_sums(2)
            pj.reconstruct(alg, 2, sino, x)
            den.append(pj.column_sums().cpu().numpy())
        out.append(x.cpu().numpy())
    assert np.array_equal(den[0].view(np.int32), den[1].view(np.int32))
    assert np.array_equal(out[0].view(np.int32), out[1].view(np.int32))
