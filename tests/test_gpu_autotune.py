"""The autotuner times what can differ: every (lanes, bundle) pair where the
projections take the whole-ray form, which reads them, one pair where they take
another form, and a stack's last slices with and without a launch of their own.
What it sets is among what it timed and keeps the sums."""
import numpy as np
import pytest

from trace_amd.phantom import angles_rad

pytestmark = pytest.mark.gpu


def _tune(torch, N, P, S, staged=None, **kw):
    from trace_amd import Projector
    from trace_amd.autotune import autotune
    th = angles_rad(P)
    gen = torch.Generator(device="cuda").manual_seed(S)
    sino = torch.rand((P, S, N), generator=gen, device="cuda") + 0.5
    x = torch.ones((S, N, N), device="cuda")
    pj = Projector(th, S, N, N / 2.0 + 0.3)
    if staged is not None:
        pj.set_fwd_staged(staged)
    return pj, autotune(pj, sino, x, "mlem", **kw), sino


def _pairs(res, fb):
    return {tuple(map(int, k.split("x")[1:])) for k in res["forward_ms"] if k.startswith(f"{fb}x")}


def test_whole_ray_pairs_are_all_timed(gpu):
    """32 slices whose projections take whole rays: the default pair (4, 16)
    is among the candidates."""
    import torch
    from trace_amd import _capi
    from trace_amd.autotune import FWD_SHAPES
    pj, res, _ = _tune(torch, 80, 60, 32, fwd_batches=(4, 32), tiles=((16, 16, 32),))
    with pj:
        assert _pairs(res, 32) == {(ln, ba) for fb, ln in FWD_SHAPES if fb == 32
                                   for ba in (1, 2, 4, 8, 16)}
        assert (4, 16) in _pairs(res, 32)
        assert _pairs(res, 4) == {(1, 8)}  # several lanes share a ray: one launch
        fb, ln, ba = min(res["forward_ms"], key=res["forward_ms"].get).split("x")
        assert pj.launch_shape()[0] == int(fb)
        assert (pj.fwd_lanes(), pj.fwd_bundle()) == (int(ln), int(ba))
        if int(fb) == 32:
            assert pj.fwd_form() == _capi.TRACE_FORM_WHOLE


@pytest.mark.parametrize("S,fb,pair", [(32, 32, (4, 16)), (16, 16, (2, 8)), (4, 4, (1, 8))])
def test_staged_batches_are_timed_once(gpu, S, fb, pair):
    import torch
    from trace_amd import _capi
    pj, res, _ = _tune(torch, 96, 60, S, staged=True, fwd_batches=(fb,), tiles=((16, 16, fb),))
    with pj:
        assert pj.fwd_form() == _capi.TRACE_FORM_STAGED
        assert _pairs(res, fb) == {pair}


@pytest.mark.parametrize("S", [33, 64])
def test_last_slices(gpu, S):
    import torch
    from trace_amd import Projector, _capi
    from trace_amd.autotune import apply_shape
    N, P = 256, 20
    pj, res, sino = _tune(torch, N, P, S, fwd_batches=(32,), tiles=((16, 16, 32),))
    timed = {k: v for k, v in res["back_ms"].items()}
    assert set(timed) == ({"16x16x32", "16x16x32+rest"} if S == 33 else {"16x16x32"})
    if S == 33:
        assert res["rest"] == (timed["16x16x32+rest"] < timed["16x16x32"])
    else:
        assert res["rest"]  # nothing to time: as a new handle
    z = []
    with pj:
        assert pj.get_option(_capi.TRACE_OPT_BACK_REST) == int(res["rest"])
        for rest in (False, True):
            apply_shape(pj, dict(res, rest=rest))
            assert pj.get_option(_capi.TRACE_OPT_BACK_REST) == int(rest)
            z.append(pj.adjoint(sino))
    with Projector(angles_rad(P), S, N, N / 2.0 + 0.3) as pj:
        assert pj.get_option(_capi.TRACE_OPT_BACK_REST) == 1
        z.append(pj.adjoint(sino))
        pj.set_launch_shape(32, 16, 16, 32)
        assert pj.get_option(_capi.TRACE_OPT_BACK_REST) == 0
    assert torch.equal(z[0], z[1]) and torch.equal(z[0], z[2])


@pytest.mark.parametrize("S,batches", [(1, {1}), (2, {1, 2}), (3, {1, 2, 4}), (5, {1, 2, 4, 8})])
def test_forward_batches_fill_the_stack(gpu, S, batches):
    import torch
    pj, res, _ = _tune(torch, 48, 20, S, bundles=(8,), tiles=((16, 16, 4),))
    with pj:
        assert {int(k.split("x")[0]) for k in res["forward_ms"]} == batches


def test_form_is_read_only(gpu):
    from trace_amd import Projector, _capi
    with Projector(angles_rad(8), 4, 16, 8.0) as pj:
        assert pj.fwd_form() == _capi.TRACE_FORM_SPLIT
        L = _capi.lib()
        assert (L.trace_set_option(pj.handle, _capi.TRACE_OPT_FWD_FORM, 0)
                == _capi.TRACE_E_UNSUPPORTED)
        assert (L.trace_set_option(pj.handle, _capi.TRACE_OPT_BACK_REST, 2)
                == _capi.TRACE_E_INVALID)
