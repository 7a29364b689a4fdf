"""Performance cases: the work that programs have this package do.

A case is one call (or one training step) through the public entry points:
`Projector` (device reconstruction, forward projection, adjoint), the
application-level calls on host arrays, `Batch` and the differentiable ray
transform.  `listed()` holds the named cases, `draw(rng)` makes one more of
the same ranges: images of 48 to 2048 pixels a side, 30 to 1500 angles, 1 to
64 slices, all four algorithms, image sides that differ from the detector
width, off-centre rotation axes, either rounding of the segment lengths.

`exact(case, seed)` evaluates the same products in float64.  The discrete
operator is defined by single-precision crossing coordinates (a source point
10^6 pixels away: trace_utils.cc:48-187), so those are formed in float32, and
lengths, sums and updates in float64 (`SystemMatrix`).
"""
from __future__ import annotations

import ctypes
import ctypes.util
import math

import numpy as np
import torch

DEVICE = "cuda:0"


# ------------------------------------------------------------------ cases --

def _case(op, name=None, **kw):
    c = {"op": op, "alg": "", "slices": 1, "side": 256, "cols": 0, "angles": 180, "iters": 1,
         "offset": 0.0, "hardware_sqrt": False, "specs": ""}
    c.update(kw)
    if not c["cols"]:
        c["cols"] = c["side"]
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: one forward projection of a small slice inside
        # an interactive or per-slice loop, where launches and host work count
        _case("forward", "forward_1x64_48", side=64, angles=48),
        # one slice of the smallest reference configuration, a whole
        # reconstruction: 20 iterations of three short kernels each
        _case("reconstruct", "sirt_1x256_180_20it", alg="sirt", side=256, angles=180, iters=20),
        # one slice at a usual detector size, the iteration loop of a
        # slice-by-slice program
        _case("reconstruct", "mlem_1x1024_720_5it", alg="mlem", side=1024, angles=720, iters=5),
        # a few slices of odd sizes with an off-centre axis (a cropped
        # detector): the adjoint alone, as a solver outside calls it
        _case("adjoint", "adjoint_5x725_401", slices=5, side=725, angles=401, offset=1.7),
        # a dozen slices with an image smaller than the detector, hardware
        # square roots: a preview reconstruction
        _case("reconstruct", "sirt_12x600_361_2it", alg="sirt", slices=12, side=600, cols=768,
              angles=361, iters=2, offset=-2.3, hardware_sqrt=True),
        # the benchmark's stack: 64 slices of 2048^2 resident in HBM, one
        # iteration of a long loop
        _case("reconstruct", "mlem_64x2048_1500_1it", alg="mlem", slices=64, side=2048,
              angles=1500),
        # regularised reconstruction of a stack (sums in the reference's
        # order), the second benchmark configuration at a quarter of its size
        _case("reconstruct", "pml_32x1024_720_2it", alg="pml", slices=32, side=1024, angles=720,
              iters=2),
        # 3-D regularisation of a thin stack with odd sizes
        _case("reconstruct", "apmlr_9x511_363_3it", alg="apmlr", slices=9, side=511, angles=363,
              iters=3),
        # uneven slices (every slice its own geometry) in one graph launch
        _case("batch", "batch_16_uneven_2it", iters=2,
              specs="256:180 1024:901 512:400 2048:600 1536:1111 256:959 512:1800 1024:333 "
                    "300:500 1024:720 256:1500 725:640 512:241 1536:422 2048:350 1024:1234"),
        # one step of regularised least squares through autograd: loss,
        # forward and backward projection, total variation
        _case("gradient", "gradient_1x2048_1500", side=2048, angles=1500),
        # the differentiable unrolled solver as a training layer, small
        # images, forward and backward
        _case("unrolled", "unrolled_1x320_256_4it", side=320, angles=256, iters=4),
        # what the reconstruction programs do with a dataset in host memory:
        # geometry tables, column sums, copies and iterations in one call
        _case("host", "host_mlem_4x640_480_10it", alg="mlem", slices=4, side=640, angles=480,
              iters=10),
    ]


def _cost(c):
    """Segment-slices of one pass, with the walks shared by up to 32 slices."""
    if c["op"] == "batch":
        return sum(n * n * p for n, p in _specs(c)) * c["iters"] * 26
    walks = -(-c["slices"] // 32) * 24 + c["slices"] * 2
    return c["side"] * min(c["side"], c["cols"]) * c["angles"] * c["iters"] * walks


_LARGEST = 2048 * 2048 * 1500 * (2 * 24 + 64 * 2)


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["forward", "adjoint", "reconstruct", "reconstruct", "reconstruct",
                     "reconstruct", "batch", "gradient", "unrolled", "host"])
    while True:
        c = _case(op, side=_log_uniform(rng, 48, 2048), angles=_log_uniform(rng, 30, 1500),
                  offset=round(rng.uniform(-4.0, 4.0), 1))
        if op in ("forward", "adjoint", "reconstruct", "host"):
            c["slices"] = _log_uniform(rng, 1, 64)
        if op in ("reconstruct", "host"):
            c["alg"] = rng.choice(["sirt", "mlem", "pml", "apmlr"])
        if op in ("reconstruct", "host", "unrolled"):
            c["iters"] = rng.randint(1, 6 if op == "unrolled" else 10)
        if op in ("forward", "adjoint", "reconstruct"):
            if rng.random() < 0.25:
                c["cols"] = max(32, int(c["side"] * rng.uniform(0.7, 1.4)))
                if c["alg"] in ("pml", "apmlr"):
                    c["cols"] = c["side"]
            c["hardware_sqrt"] = rng.random() < 0.15
        if op == "batch":
            c["iters"] = rng.randint(1, 4)
            c["specs"] = " ".join(
                f"{rng.choice([256, 300, 512, 725, 1024, 1536])}:{rng.randint(180, 1200)}"
                for _ in range(rng.randint(3, 14)))
        if _cost(c) <= 0.5 * _LARGEST:
            return c


def _specs(c):
    return [tuple(int(v) for v in s.split(":")) for s in c["specs"].split()]


def _center(side_cols, offset):
    return side_cols / 2.0 + offset


# ------------------------------------------------------------------ inputs --

def _theta(P):
    from trace_amd.phantom import angles_rad
    return angles_rad(P)


def _sinogram(theta, C, S, seed, offset):
    """Poisson-noisy line integrals of ellipse phantoms [P][S][C]."""
    from trace_amd.phantom import noisy_sinogram
    return noisy_sinogram(theta, C, S, seed=seed, I0=1e4, K=6, center=_center(C, offset),
                          device=DEVICE)


def _images(N, S, seed):
    """Ellipse phantoms on a positive background [S][N][N]."""
    from trace_amd.phantom import phantom_slices
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    x = phantom_slices(N, S, seed=seed, K=6, device=DEVICE)
    return x + 0.05 * torch.rand(x.shape, generator=gen, device=DEVICE)


def _inputs(c, seed):
    """The tensors a program has in hand before the call."""
    if c["op"] == "batch":
        out = []
        for i, (C, P) in enumerate(_specs(c)):
            th = _theta(P)
            out.append((th, _sinogram(th, C, 1, seed * 64 + i, 0.0)[:, 0, :].contiguous(),
                        ("sirt", "mlem")[i % 2]))
        return {"slices": out}
    N, C, P, S = c["side"], c["cols"], c["angles"], c["slices"]
    th = _theta(P)
    d = {"theta": th}
    if c["op"] in ("reconstruct", "host"):
        d["sino"] = _sinogram(th, C, S, seed, c["offset"])
        d["x0"] = 0.0 if c["alg"] == "sirt" else 1.0
    elif c["op"] == "forward":
        d["x"] = _images(N, S, seed)
    elif c["op"] == "adjoint":
        gen = torch.Generator(device=DEVICE)
        gen.manual_seed(seed)
        d["r"] = torch.randn((P, S, C), generator=gen, device=DEVICE)
    else:
        d["sino"] = _sinogram(th, C, 1, seed, c["offset"])[:, 0, :].contiguous()
        d["x"] = 0.5 * _images(N, 1, seed + 1)[0]
    return d


TV_WEIGHT = 1e-3
PML_BETA = 10.0


def prepare(case, seed):
    from trace_amd import Projector
    from trace_amd.autograd import RayTransform
    from trace_amd.batch import Batch, BatchSlice
    c = case
    st = {"case": c, **_inputs(c, seed)}
    if c["op"] == "batch":
        st["x"] = [torch.empty((s.shape[1], s.shape[1]), device=DEVICE) for _, s, _ in st["slices"]]
        st["batch"] = Batch([BatchSlice(th, s, x, alg, c["iters"], s.shape[1] / 2.0)
                             for (th, s, alg), x in zip(st["slices"], st["x"])])
    elif c["op"] in ("gradient", "unrolled"):
        st["op"] = RayTransform(st["theta"], c["side"], center=_center(c["cols"], c["offset"]))
        st["x"].requires_grad_(True)
        if c["op"] == "unrolled":
            st["relax"] = torch.full((c["iters"],), 0.9, device=DEVICE, requires_grad=True)
    elif c["op"] == "host":
        st["sino"] = st["sino"].cpu().numpy()
        st["degrees"] = np.asarray(np.arange(c["angles"], dtype=np.float64) * 180.0 / c["angles"],
                                   np.float32)
    else:
        st["pj"] = Projector(st["theta"], c["slices"], c["cols"], _center(c["cols"], c["offset"]),
                             exact_sqrt=not c["hardware_sqrt"], num_grids=c["side"])
        if c["op"] == "reconstruct":
            st["recon"] = torch.empty((c["slices"], c["side"], c["side"]), device=DEVICE)
    return st


def run(state):
    c = state["case"]
    op = c["op"]
    if op == "forward":
        return state["pj"].forward(state["x"])
    if op == "adjoint":
        return state["pj"].adjoint(state["r"])
    if op == "reconstruct":
        state["recon"].fill_(state["x0"])
        return state["pj"].reconstruct(c["alg"], c["iters"], state["sino"], state["recon"])
    if op == "batch":
        for x, (_, _, alg) in zip(state["x"], state["slices"]):
            x.fill_(0.0 if alg == "sirt" else 1.0)
        state["batch"].run()
        return state["x"]
    if op == "gradient":
        from trace_amd.autograd import ls_tv_loss
        x = state["x"]
        x.grad = None
        loss = ls_tv_loss(state["op"], x, state["sino"], TV_WEIGHT)
        loss.backward()
        return loss.detach(), x.grad
    if op == "unrolled":
        from trace_amd.autograd import sirt_unrolled
        x, relax = state["x"], state["relax"]
        x.grad = relax.grad = None
        y = sirt_unrolled(state["op"], state["sino"], c["iters"], x0=x, relax=relax)
        (0.5 * (y * y).sum()).backward()
        return y.detach(), x.grad, relax.grad
    return _host_call(c, state)


def _host_call(c, state):
    import trace_amd
    ctr = _center(c["cols"], c["offset"])
    if c["alg"] == "pml":  # takes radians
        return trace_amd.pml(state["theta"], state["sino"], c["iters"], ctr)
    f = {"sirt": trace_amd.sirt, "mlem": trace_amd.mlem, "apmlr": trace_amd.apmlr}[c["alg"]]
    return f(state["degrees"], state["sino"], c["iters"], ctr)


# -------------------------------------------------------------------- work --

def _work(N, C, P, S, iters, products, image_arrays, sino_arrays):
    nnz = 1.2 * N * min(N, C) * P  # segments of one slice's rays
    return {"bytes": 4.0 * iters * S * (image_arrays * N * N + sino_arrays * P * C),
            "flops": 2.0 * nnz * S * products * iters}


def work(case):
    c = case
    if c["op"] == "batch":
        w = [_work(C, C, P, 1, c["iters"], 2, 2, 1) for C, P in _specs(c)]
        return {k: sum(v[k] for v in w) for k in ("bytes", "flops")}
    N, C, P, S = c["side"], c["cols"], c["angles"], c["slices"]
    if c["op"] in ("forward", "adjoint"):
        return _work(N, C, P, S, 1, 1, 1, 1)
    if c["op"] == "gradient":
        return _work(N, C, P, 1, 1, 2, 2, 1)
    if c["op"] == "unrolled":  # forward, and its transpose backward
        return _work(N, C, P, 1, c["iters"], 4, 4, 2)
    return _work(N, C, P, S, c["iters"], 2, 2, 1)


# ------------------------------------------------------------------- exact --

def _libm(name, theta):
    """sinf or cosf of the host's C library: one unit in the last place moves
    a ray by 0.06 pixels, so the operator is defined by its values."""
    fn = getattr(ctypes.CDLL(ctypes.util.find_library("m") or "libm.so.6"), name)
    fn.restype, fn.argtypes = ctypes.c_float, [ctypes.c_float]
    return np.array([fn(float(t)) for t in np.asarray(theta, np.float32)], np.float32)


class SystemMatrix:
    """The discrete operator of one slice, as sorted crossings of every ray
    with the grid lines (angles in [0, pi)): pixel index and float64 length of
    every segment."""

    def __init__(self, theta, N, C, center, hold):
        f = np.float32
        mov = f(np.float64(f(C)) / 2.0 - np.float64(f(center)))
        if np.float64(f(mov - np.ceil(mov))) < 1e-6:
            mov = f(np.float64(mov) + 1e-6)
        yi = ((1 - C) / 2.0 + np.arange(C, dtype=np.float64) + np.float64(mov)).astype(f)
        s, co = _libm("sinf", theta)[:, None], _libm("cosf", theta)[:, None]
        xi, yi = f(-1e6), yi[None, :]
        xc, ys, xs, yc = xi * co, yi * s, xi * s, yi * co
        sx, sy = xc - ys, xs + yc
        with np.errstate(divide="ignore", invalid="ignore"):
            slope = (sy - (-xs + yc)) / (sx - -(xc + ys))
            islope = f(1.0) / slope
        # rows are walked upwards in the first quadrant, else downwards
        # (trace_utils.cc:41-46, 175-197), which decides among equal crossings
        pi = f(3.14159265358979)
        up = (np.asarray(theta, f) < pi / f(2))[:, None]
        flat = [torch.from_numpy(np.array(np.broadcast_to(v, sx.shape))).reshape(-1, 1).to(DEVICE)
                for v in (sx, sy, slope, islope, up)]
        self.N, self.rays = N, sx.size
        self.sx, self.sy, self.k, self.ik, self.up = flat
        self.chunk = max(1, int(6e7) // (2 * N + 2))
        self.parts = list(self._parts()) if hold else None

    def _parts(self):
        N = self.N
        gl = (torch.arange(N + 1, device=DEVICE, dtype=torch.float64) - N / 2.0).float()[None, :]
        half = float(np.float32(N / 2.0))
        inf = float("inf")
        for a in range(0, self.rays, self.chunk):
            e = slice(a, min(a + self.chunk, self.rays))
            rows = torch.where(self.up[e], gl, gl.flip(1))
            ax = self.ik[e] * (rows - self.sy[e]) + self.sx[e]
            by = self.k[e] * (gl - self.sx[e]) + self.sy[e]
            ina, inb = (ax > -half) & (ax < half), (by > -half) & (by < half)
            x = torch.cat([torch.where(inb, gl.expand_as(by), torch.full_like(by, inf)),
                           torch.where(ina, ax, torch.full_like(ax, inf))], 1)
            y = torch.cat([by, rows], 1)
            x, o = torch.sort(x, dim=1, stable=True)
            y = torch.gather(y, 1, o)
            ok = torch.isfinite(x[:, 1:])
            dx, dy = (x[:, 1:] - x[:, :-1])[ok], (y[:, 1:] - y[:, :-1])[ok]
            ix = (((x[:, 1:] + x[:, :-1]) * 0.5)[ok] + half).to(torch.int64)
            iy = (((y[:, 1:] + y[:, :-1]) * 0.5)[ok] + half).to(torch.int64)
            idx = ix + iy * N
            ray = torch.arange(e.start, e.stop, device=DEVICE)[:, None].expand_as(ok)[ok]
            ln = torch.sqrt(dx.double() ** 2 + dy.double() ** 2)
            keep = idx < N * N
            yield (idx[keep].to(torch.int32), ray[keep].to(torch.int32), ln[keep])

    def segments(self):
        return self.parts if self.parts is not None else self._parts()

    def forward(self, x):
        y = torch.zeros(self.rays, dtype=torch.float64, device=DEVICE)
        for i, r, ln in self.segments():
            y.index_add_(0, r, x.reshape(-1)[i] * ln)
        return y

    def adjoint(self, r_, power=1):
        z = torch.zeros(self.N * self.N, dtype=torch.float64, device=DEVICE)
        for i, r, ln in self.segments():
            z.index_add_(0, i, r_.reshape(-1)[r] * ln)
        return z

    def square_sums(self):
        a = torch.zeros(self.rays, dtype=torch.float64, device=DEVICE)
        for _, r, ln in self.segments():
            a.index_add_(0, r, ln * ln)
        return a


def _safe_div(a, b):
    return torch.where(b != 0, a / torch.where(b != 0, b, torch.ones_like(b)),
                       torch.zeros_like(a))


def _stencil(x, inter, beta, beta1, delta, delta1, regw):
    """F and G of the regularised updates (pml.cc:25-201, apmlr.cc:919-982)
    for a stack [S][N][N]; `inter` adds the weights and neighbours across
    slices, without it the in-plane weights carry no edge term."""
    S, N, _ = x.shape
    ones = torch.ones((N, N), dtype=torch.float64, device=x.device)
    offs = [(1, 0), (-1, 0), (0, 1), (0, -1), (1, 1), (-1, 1), (1, -1), (-1, -1)]

    def shifted(v, dx, dy):
        out = torch.zeros_like(v)
        H, W = v.shape[-2:]
        out[..., max(0, -dy):H - max(0, dy), max(0, -dx):W - max(0, dx)] = \
            v[..., max(0, dy):H + min(0, dy), max(0, dx):W + min(0, dx)]
        return out

    has = [shifted(ones, dx, dy) for dx, dy in offs]
    base = sum(h * (1.0 if k < 4 else 1 / math.sqrt(2.0)) for k, h in enumerate(has))
    F, G = torch.zeros_like(x), torch.zeros_like(x)
    for s in range(S):
        zs = []
        if inter:
            zs = [1] if s == 0 else ([-1] if s == S - 1 else [1, -1])
        total = base + len(zs) * regw
        for k, (dx, dy) in enumerate(offs):
            xq = shifted(x[s], dx, dy)
            w = has[k] * (1.0 if k < 4 else 1 / math.sqrt(2.0)) / total
            g = 1.0 / (1.0 + ((x[s] - xq) / delta).abs()) if inter else 1.0
            F[s] += 2 * beta * w * g
            G[s] -= 2 * beta * w * g * (x[s] + xq)
        for dz in zs:
            xq = x[s + dz] if 0 <= s + dz < S else torch.ones_like(x[s])
            g = 1.0 / (1.0 + ((x[s] - xq) / delta1).abs())
            F[s] += 2 * beta1 * regw / total * g
            G[s] -= 2 * beta1 * regw / total * g * (x[s] + xq)
    return F, G


def _reconstruct(A, sino, alg, iters, x0, S):
    """The iterations in float64; sino [S][rays]."""
    N = A.N
    x = torch.full((S, N, N), x0, dtype=torch.float64, device=DEVICE)
    den = A.adjoint(torch.ones(A.rays, dtype=torch.float64, device=DEVICE)).reshape(N, N)
    a2 = A.square_sums() if alg == "sirt" else None
    for _ in range(iters):
        if alg in ("sirt", "mlem"):
            for s in range(S):
                y = A.forward(x[s])
                if alg == "sirt":
                    x[s] += A.adjoint(_safe_div(sino[s] - y, a2)).reshape(N, N) / den
                else:
                    x[s] *= A.adjoint(_safe_div(sino[s], y)).reshape(N, N) / den
            continue
        # the ray pass of an APMLR slice reads the slice below it, the first
        # one a constant 1 (apmlr.cc:1082-1084)
        src = x if alg == "pml" else torch.cat([torch.ones_like(x[:1]), x[:-1]])
        F, G = _stencil(x, alg == "apmlr", PML_BETA, 1.0, 1.0, 1.0, 1.0)
        new = torch.empty_like(x)
        for s in range(S):
            num = -src[s] * A.adjoint(_safe_div(sino[s], A.forward(src[s]))).reshape(N, N)
            g = G[s] + den
            new[s] = (-g + torch.sqrt(g * g - 8 * num * F[s])) / (4 * F[s])
        x = new
    return x


def _points(N, C, P):
    return float(P) * C * (2 * N + 2)


def exact(case, seed):
    c = case
    d = None
    if c["op"] == "batch":
        out = []
        d = _inputs(c, seed)
        for th, s, alg in d["slices"]:
            C, P = s.shape[1], s.shape[0]
            if _points(C, C, P) > 3e8:
                out.append(None)
                continue
            A = SystemMatrix(th, C, C, C / 2.0, True)
            out.append(_reconstruct(A, s.double().reshape(1, -1), alg, c["iters"],
                                    0.0 if alg == "sirt" else 1.0, 1)[0].cpu())
        return out
    N, C, P, S = c["side"], c["cols"], c["angles"], c["slices"]
    pts = _points(N, C, P)
    products = S * max(1, c["iters"]) * (4 if c["op"] == "unrolled" else 2) + 2
    hold = pts <= 2.5e9
    if pts > 2e10 or (not hold and products > 4) or pts * products > 4e10:
        return None
    d = _inputs(c, seed)
    ctr = _center(C, c["offset"])
    th = d["theta"]
    if c["op"] == "host" and c["alg"] == "apmlr" and S == 1:
        return None
    A = SystemMatrix(th, N, C, ctr, hold)
    if c["op"] == "forward":
        return torch.stack([A.forward(x.double()).reshape(P, C) for x in d["x"]], 1).cpu()
    if c["op"] == "adjoint":
        r = d["r"].double().permute(1, 0, 2).reshape(S, -1)
        return torch.stack([A.adjoint(v).reshape(N, N) for v in r]).cpu()
    if c["op"] in ("reconstruct", "host"):
        sino = d["sino"].double().permute(1, 0, 2).reshape(S, -1)
        if c["alg"] != "sirt":
            sino = sino.abs()
        return _reconstruct(A, sino, c["alg"], c["iters"], d["x0"], S).cpu()
    sino, x = d["sino"].double().reshape(-1), d["x"].double()
    if c["op"] == "gradient":
        from torch.nn.functional import pad
        r = A.forward(x) - sino
        dx = pad(x[:, 1:] - x[:, :-1], (0, 1))
        dy = pad(x[1:, :] - x[:-1, :], (0, 0, 0, 1))
        n = torch.sqrt(dx * dx + dy * dy + 1e-8)
        px, py = dx / n, dy / n
        g = -(px + py) + pad(px[:, :-1], (1, 0)) + pad(py[:-1, :], (0, 0, 1, 0))
        loss = 0.5 * (r * r).sum() + TV_WEIGHT * n.sum()
        return loss.cpu(), (A.adjoint(r).reshape(N, N) + TV_WEIGHT * g).cpu()
    # unrolled: x_{k+1} = x_k + relax_k inv_den A^T((p - A x_k) / a2)
    relax = 0.9
    a2 = A.square_sums()
    ia2 = _safe_div(torch.ones_like(a2), torch.where(a2 > 0, a2, torch.ones_like(a2)))
    den = A.adjoint(torch.ones_like(a2)).reshape(N, N)
    inv = torch.where(den > 0, 1.0 / den, torch.zeros_like(den))
    steps = []
    for _ in range(c["iters"]):
        u = A.adjoint((sino - A.forward(x)) * ia2).reshape(N, N) * inv
        steps.append(u)
        x = x + relax * u
    g, gr = x.clone(), []
    for u in reversed(steps):
        gr.insert(0, (g * u).sum())
        g = g - relax * A.adjoint(A.forward(g * inv) * ia2).reshape(N, N)
    return x.cpu(), g.cpu(), torch.stack(gr).cpu()
