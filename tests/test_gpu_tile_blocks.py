"""The tile backprojector's workgroup sizes (256, 512 and 1024 lanes, chosen
by how many tiles the launch has) and the slices' rounding constants.  Its
sums are integers, so every tile shape and workgroup size must give the same
bits, and scaling the input by a power of two must scale the output by it,
also past the exponents the all-fixed form covers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# slices -> tile shapes of that stack
SHAPES = {
    1: [(16, 16, 1), (32, 32, 1), (64, 64, 1), (64, 64, 2), (8, 8, 16)],
    5: [(16, 16, 4), (32, 32, 4), (16, 16, 8), (24, 24, 8), (32, 32, 8), (16, 32, 8)],
    35: [(16, 16, 16), (32, 32, 16), (32, 16, 16), (16, 16, 32), (8, 8, 16)],
}


@pytest.mark.parametrize("S", [1, 5, 35])
@pytest.mark.parametrize("N,P,center", [(90, 31, 45.0), (520, 14, 259.3), (1100, 6, 550.5)])
def test_shapes_and_blocks_bit_identical(gpu, N, P, center, S):
    torch = gpu
    from trace_amd import Projector
    rng = np.random.default_rng(N + S)
    th = rng.uniform(0, np.pi, P).astype(np.float32)
    r = torch.from_numpy(rng.normal(size=(P, S, N)).astype(np.float32)).cuda()
    want = None
    with Projector(th, S, N, center) as pj:
        for tw, th_, tb in SHAPES[S]:
            print(f"tile {tw}x{th_}x{tb} N={N} P={P} S={S}", flush=True)
            pj.set_launch_shape(1, tw, th_, tb)
            z = pj.adjoint(r).cpu().numpy()
            want = z if want is None else want
            assert np.array_equal(z.view(np.int32), want.view(np.int32)), (tw, th_, tb)


@pytest.mark.parametrize("S", [1, 3, 20])
@pytest.mark.parametrize("e", [-124, -112, -60, 60, 104])
def test_power_of_two_scaling(gpu, S, e):
    """z(2^e r) = 2^e z(r), for inputs whose scale exponents lie inside and
    outside the range of the rounding constants (results below the normal
    floats are left out)."""
    torch = gpu
    from trace_amd import Projector
    N, P = 80, 40
    rng = np.random.default_rng(S)
    th = rng.uniform(0, np.pi, P).astype(np.float32)
    r = rng.uniform(0.5, 1.0, (P, S, N)).astype(np.float32)
    with Projector(th, S, N, N / 2.0) as pj:
        z0 = pj.adjoint(torch.from_numpy(r).cuda()).cpu().numpy()
        z1 = pj.adjoint(torch.from_numpy(np.ldexp(r, e)).cuda()).cpu().numpy()
    ok = np.abs(z0.astype(np.float64)) * 2.0 ** e >= 2.0 ** -126
    assert ok.mean() > 0.9
    assert np.array_equal(np.ldexp(z0, e)[ok].view(np.int32), z1[ok].view(np.int32))
