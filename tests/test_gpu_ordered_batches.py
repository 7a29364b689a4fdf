"""Ordered sums over the slice batches the library chooses.

The tile form takes 1 to 32 slices a thread, by the stack and by the number of
image tiles; the per-pixel form takes at most 8 and shares none of its code
for the sums.  Both add every pixel's segments in the same order, so their
images are equal bit for bit, whatever the batch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (N, S): 328 has 41 x 41 tiles of 8 x 8, enough for the deepest batch a stack
# allows; 72 has 81, which takes shallow ones; 17 has a partial last tile
SIZES = [(328, 1), (328, 3), (328, 7), (328, 12), (328, 20), (328, 33),
         (200, 9), (72, 33), (17, 40)]


def _image(alg, th, sino, init, N, tile):
    import torch
    from trace_amd import Projector, RegParams
    _, S, C = sino.shape
    with Projector(th, S, C, C / 2, num_grids=N) as pj:
        pj.set_ordered_sums(2)
        pj.set_ordered_tile(tile)
        ds = torch.from_numpy(sino).cuda()
        dx = torch.from_numpy(init).cuda()
        pj.reconstruct(alg, 1, ds, dx, RegParams())
        torch.cuda.synchronize()
        return dx.cpu().numpy()


@pytest.mark.parametrize("alg", ["mlem", "pml"])
@pytest.mark.parametrize("N,S", SIZES)
def test_tile_form_equals_pixel_form(gpu, alg, N, S):
    from trace_amd.phantom import angles_rad
    P = 14
    rng = np.random.default_rng(N + S)
    th = angles_rad(P)
    sino = rng.uniform(0.1, 2.0, (P, S, N)).astype(np.float32)
    init = rng.uniform(0.5, 1.5, (S, N, N)).astype(np.float32)
    print(f"ordered {alg} N={N} S={S}", flush=True)
    a = _image(alg, th, sino, init, N, True)
    b = _image(alg, th, sino, init, N, False)
    bad = int(np.count_nonzero(a.view(np.uint32) != b.view(np.uint32)))
    assert bad == 0, f"{bad} of {a.size} pixels differ"
