"""Every form of the forward projector against the oracle, at sizes that select
it: the whole-ray form at each compiled slice batch and lanes per ray, and the
form with several lanes per ray at four lanes (eight: test_gpu_split.py).  Ray
sums bit for bit; SIRT and MLEM with every sum in the reference's order, bit for
bit as well (the weights), and with the default sums against another form (the
weights' maxima, which set the fixed-point scale)."""
import numpy as np
import pytest

from trace_amd.phantom import angles_rad

pytestmark = pytest.mark.gpu

WHOLE, STAGED, SPLIT = 0, 1, 2

# slice batch, slices, angles (64 columns): more rays than the form with several
# lanes per ray takes at that batch (split_lanes)
WHOLE_SIZES = {1: (1, 7820), 2: (2, 3910), 4: (3, 1570), 8: (7, 205), 16: (13, 103), 32: (21, 53)}
WHOLE_FORMS = [(1, 1, 8), (1, 1, 16), (2, 1, 4), (4, 1, 2), (8, 1, 16), (8, 2, 8), (16, 1, 1),
               (16, 2, 8), (16, 4, 1), (16, 4, 8), (32, 1, 8), (32, 2, 16), (32, 4, 16)]
# slices of a batch of 2, 4 and 8 and angles (70 columns): four lanes per ray
SPLIT_SIZES = [(2, 1400), (3, 1000), (8, 90)]


def _bits(a):
    return np.asarray(a, np.float32).view(np.int32)


def _form(pj):
    from trace_amd import _capi
    return pj.get_option(_capi.TRACE_OPT_FWD_FORM)


@pytest.mark.parametrize("fb,lanes,ba", WHOLE_FORMS)
def test_whole_ray_sums(gpu, oracle, fb, lanes, ba):
    import torch
    from trace_amd import Projector
    N = 64
    S, P = WHOLE_SIZES[fb]
    th = np.random.default_rng(fb * lanes + ba).uniform(-1, 4, P).astype(np.float32)
    x = np.random.default_rng(ba).uniform(0, 1, (S, N, N)).astype(np.float32)
    with Projector(th, S, N, N / 2.0 + 0.5) as pj:
        pj.set_fwd_bundle(1)
        pj.set_launch_shape(fb, 16, 16, 8)
        pj.set_fwd_lanes(lanes)
        pj.set_fwd_bundle(ba)
        pj.set_fwd_staged(False)
        assert _form(pj) == WHOLE
        y = pj.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    assert np.array_equal(_bits(y), _bits(oracle.forward(th, x, N / 2.0 + 0.5)))


@pytest.mark.parametrize("S,P", SPLIT_SIZES)
def test_four_lane_sums(gpu, oracle, S, P):
    import torch
    from trace_amd import Projector
    N = 70
    th = np.concatenate([angles_rad(P - 5), np.float32([-0.4, -2.1, -3.0, 3.7, 5.5])])
    x = np.random.default_rng(S).standard_normal((S, N, N)).astype(np.float32)
    with Projector(th, S, N, N / 2.0 + 0.5) as pj:
        assert _form(pj) == SPLIT
        y = pj.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    assert np.array_equal(_bits(y), _bits(oracle.forward(th, x, N / 2.0 + 0.5)))


def _recon(alg, th, sino, center, staged=None, ordered=None):
    import torch
    from trace_amd import Projector
    P, S, N = sino.shape
    x = torch.full((S, N, N), 0.0 if alg == "sirt" else 1.0, device="cuda:0")
    with Projector(th, S, N, center) as pj:
        if staged is not None:
            pj.set_fwd_staged(staged)
        if ordered is not None:
            pj.set_ordered_sums(ordered)
        form = _form(pj)
        pj.reconstruct(alg, 2, torch.from_numpy(np.ascontiguousarray(sino)).cuda(), x)
    return x.cpu().numpy(), form


@pytest.mark.parametrize("alg", ["sirt", "mlem"])
@pytest.mark.parametrize("form,S,P", [(WHOLE, 3, 1570), (WHOLE, 7, 205), (WHOLE, 13, 103),
                                      (SPLIT, 2, 1400), (SPLIT, 3, 1000), (SPLIT, 8, 90),
                                      (STAGED, 3, 60), (STAGED, 7, 75), (STAGED, 13, 64),
                                      (STAGED, 16, 37)])
def test_weights(gpu, oracle, alg, form, S, P):
    N = 64
    th = angles_rad(P)
    center = N / 2.0 + 0.7
    sino = np.random.default_rng(P).uniform(0.5, 2.0, (P, S, N)).astype(np.float32)
    x, got = _recon(alg, th, sino, center, form == STAGED, ordered=2)
    assert got == form
    init = np.full((S, N, N), 0.0 if alg == "sirt" else 1.0, np.float32)
    want = oracle.reconstruct(alg, th, sino, init, center, 2)
    assert np.array_equal(_bits(x), _bits(want))


@pytest.mark.parametrize("alg", ["sirt", "mlem"])
@pytest.mark.parametrize("form,S,P", [(SPLIT, 2, 1400), (SPLIT, 3, 1000), (SPLIT, 8, 90),
                                      (WHOLE, 3, 1570), (WHOLE, 7, 205), (WHOLE, 13, 103)])
def test_maxima_as_in_a_deep_stack(gpu, alg, form, S, P):
    """The default (fixed-point) sums: the same bits as the slices have in a
    stack of 21, whose projections take the whole-ray form at 32 slices."""
    N = 64
    th = angles_rad(P)
    sino = np.random.default_rng(P).uniform(0.5, 2.0, (P, 21, N)).astype(np.float32)
    sino *= np.ldexp(1.0, np.arange(21) % 7 - 3).astype(np.float32)[None, :, None]
    deep, deep_form = _recon(alg, th, sino, N / 2.0 + 0.7, False)
    x, got = _recon(alg, th, sino[:, :S], N / 2.0 + 0.7, False)
    assert got == form and deep_form == WHOLE
    assert np.array_equal(_bits(x), _bits(deep[:S]))


@pytest.mark.parametrize("alg", ["sirt", "mlem", "pml", "apmlr"])
@pytest.mark.parametrize("S", [3, 4, 7, 13, 16])
def test_staged_reconstructions(gpu, alg, S):
    """The staged form's weights and maxima at batches 4, 8 and 16, full and
    partly filled, against the other forms."""
    N, P = 96, 140
    th = angles_rad(P)
    sino = np.random.default_rng(S).uniform(0.5, 2.0, (P, S, N)).astype(np.float32)
    staged, form = _recon(alg, th, sino, N / 2.0 - 1.2, True)
    other, other_form = _recon(alg, th, sino, N / 2.0 - 1.2, False)
    assert form == STAGED and other_form == (SPLIT if S <= 4 else WHOLE)
    assert np.array_equal(_bits(staged), _bits(other))
