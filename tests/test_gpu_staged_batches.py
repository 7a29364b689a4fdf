"""Slab-staged forward projector at every compiled slice batch and slab
thickness against the whole-ray form: the same ray sums bit for bit (each
lane walks its own ray in the reference's order, sirt.cc:4-19; only the
source of its pixels differs).  The angle sets make every kind of group:
full ones, ones cut where the sweep or the column order turns round, single
angles, projections in no order, few angles (thin slabs, wide windows)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _angles(kind, P):
    from trace_amd.phantom import angles_rad
    rng = np.random.default_rng(P)
    if kind == "half turn":
        return angles_rad(P)
    if kind == "full turn":
        return (np.arange(P) * 2 * np.pi / P).astype(np.float32)
    if kind == "shuffled":
        return rng.permutation(angles_rad(P))
    return rng.uniform(-7, 7, P).astype(np.float32)


# N, C, P, centre
GEOMS = [(96, 96, 75, 48.0), (63, 70, 40, 33.2), (130, 100, 33, 50.5), (257, 257, 16, 128.5),
         (640, 640, 7, 320.0), (5, 9, 3, 4.5)]


@pytest.mark.parametrize("kind", ["half turn", "full turn", "shuffled", "any"])
@pytest.mark.parametrize("N,C,P,center", GEOMS)
@pytest.mark.parametrize("S,sb", [(3, 4), (5, 4), (7, 8), (19, 16), (33, 32)])
def test_staged_batches_bit_identical(gpu, S, sb, N, C, P, center, kind):
    import torch
    from trace_amd import Projector
    th = _angles(kind, P)
    gen = torch.Generator(device="cuda").manual_seed(S * N)
    x = torch.rand((S, N, N), generator=gen, device="cuda")
    print(f"staged S={S} batch {sb} N={N} C={C} P={P} centre={center} {kind}", flush=True)
    ys = []
    for staged in (True, False):
        with Projector(th, S, C, center, num_grids=N) as pj:
            pj.set_launch_shape(sb, 16, 16, 4)
            pj.set_fwd_staged(staged)
            ys.append(pj.forward(x).cpu().numpy())
    assert np.array_equal(ys[0].view(np.int32), ys[1].view(np.int32))


def test_form_is_chosen_until_set(gpu):
    """The option reads 1 until it is set, and the chosen form gives the same
    sums as either."""
    import torch
    from trace_amd import Projector, _capi
    from trace_amd.phantom import angles_rad
    x = torch.rand((16, 512, 512), device="cuda")
    ys = []
    for staged in (None, True, False):
        with Projector(angles_rad(200), 16, 512, 256.0) as pj:
            assert pj.get_option(_capi.TRACE_OPT_FWD_STAGED) == 1
            if staged is not None:
                pj.set_fwd_staged(staged)
            ys.append(pj.forward(x))
    assert torch.equal(ys[0], ys[1]) and torch.equal(ys[0], ys[2])
