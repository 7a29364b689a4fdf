"""Launch-shape autotuner for the forward projector and the tile
backprojector.

The forward projector's shape is its slice batch (slices gathered per
segment, 1 to 32) and, in its whole-ray form, the lanes per ray and the
ray-bundle width.  Which form a batch takes depends on the geometry
(Projector.fwd_form); the others read neither, and are timed once.  The
backprojector's shape is its image tile and slice batch (tile_w x tile_h pixels
x tile_batch slices of LDS accumulators) and, for 32-slice tiles, whether a few
slices past the last full batch take a launch of their own.  The two
kernels are independent, so each is tuned on its own: every candidate runs
one iteration of the real workload and the phase timer (HIP events on the
handle's stream) gives the kernel's time.  Results are cached per
(device name, N, P, S, algorithm).
"""
from __future__ import annotations

import json
import os

from . import _capi

FWD_BATCHES = (1, 2, 4, 8, 16, 32)
BUNDLES = (1, 2, 4, 8, 16)
TILES = ((16, 16, 8), (16, 16, 16), (16, 16, 4), (24, 24, 8), (32, 16, 8),
         (16, 32, 8), (32, 32, 4), (32, 32, 8), (8, 8, 16), (64, 64, 2),
         (32, 32, 1), (64, 64, 1), (32, 32, 2), (16, 16, 2), (16, 16, 1),
         (16, 16, 32), (32, 32, 16), (32, 16, 16), (24, 24, 16))


def _pow2_ceil(n: int) -> int:
    p = 1
    while p < n:
        p *= 2
    return p


def batch_candidates(batches, S: int):
    """Slice batches worth timing for a stack of S slices: no more than one
    batch of padding (<= max(4, S rounded up to a power of two)) and no more
    than 8 launches' worth of repeated traversal (>= S / 8)."""
    hi = max(4, _pow2_ceil(S))
    c = [b for b in batches if b <= hi and 8 * b >= S]
    return c or [max(batches)]


def forward_batches(batches, S: int):
    """Those of batch_candidates that the stack fills: a deeper one gathers
    padding, and with one slice to a batch the image needs no copy, which the
    forward projector's time does not show."""
    c = batch_candidates(batches, S)
    return [b for b in c if b <= _pow2_ceil(S)] or c[:1]


_CACHE: dict = {}


# (slice batch, lanes per ray) pairs compiled into the forward projector
FWD_SHAPES = {(1, 1), (2, 1), (4, 1), (8, 1), (16, 1), (32, 1), (8, 2), (16, 2), (32, 2),
              (16, 4), (32, 4)}
LANES = (1, 2, 4)


def _default_pair(fb: int):
    """(lanes per ray, bundle) of a new handle with slice batch fb."""
    return (4, 16) if fb == 32 else ((2, 8) if fb >= 8 else (1, 8))


def forward_pairs(pj, fb: int, lanes_per_ray=LANES, bundles=BUNDLES):
    """(lanes per ray, bundle) pairs worth timing at slice batch fb, which is
    set on `pj`: the compiled ones, or, where the projections take a form that
    reads neither, the one a new handle has (or the first)."""
    pairs = [(ln, ba) for ln in lanes_per_ray for ba in bundles
             if (fb, ln) in FWD_SHAPES and ba * ln <= 64]
    if pj.fwd_form() != _capi.TRACE_FORM_WHOLE and pairs:
        own = _default_pair(fb)
        pairs = [own if own in pairs else pairs[0]]
    return pairs


def has_rest(S: int) -> bool:
    """Whether a stack's last batch of 32 slices is at most half full."""
    return S > 32 and 1 <= S % 32 <= 16


def apply_shape(pj, res: dict):
    """Sets {"shape": (fwd_batch, tile_w, tile_h, tile_batch), "bundle",
    "lanes", "rest"} on projector `pj`."""
    pj.set_fwd_bundle(1)
    pj.set_launch_shape(*res["shape"])
    pj.set_fwd_lanes(res.get("lanes", 1))
    pj.set_fwd_bundle(res["bundle"])
    pj.set_back_rest(bool(res.get("rest", False)))


def _key(pj, alg):
    import torch
    name = torch.cuda.get_device_name(pj.device)
    return f"{name}|N{pj.N}|P{pj.P}|S{pj.S}|{alg}"


def autotune(pj, sino, recon, alg: str = "mlem", params=None,
             fwd_batches=FWD_BATCHES, bundles=BUNDLES, tiles=TILES,
             cache_file: str | None = None, verbose: bool = False,
             lanes_per_ray=LANES) -> dict:
    """Times the candidates on (sino, a copy of recon) and sets the best
    shape on projector `pj`.  Returns {"shape": (fb, tw, th, tb),
    "bundle": angles, "lanes": lanes per ray, "rest": launch of its own for
    the last slices, "forward_ms": {...}, "back_ms": {...}}."""
    import torch
    key = _key(pj, alg)
    if cache_file and not _CACHE and os.path.exists(cache_file):
        try:
            with open(cache_file) as f:
                _CACHE.update(json.load(f))
        except (OSError, ValueError):
            pass
    if key in _CACHE:
        res = _CACHE[key]
        apply_shape(pj, res)
        return res
    work = recon.clone()
    fwd_ms, back_ms = {}, {}
    tile_batches = batch_candidates(sorted({t[2] for t in tiles}), pj.S)
    base_tile = next(t for t in tiles if t[2] in tile_batches)
    pj.set_phase_timing(True)
    try:
        for fb in forward_batches(fwd_batches, pj.S):
            apply_shape(pj, {"shape": (fb, *base_tile), "bundle": 1, "lanes": 1})
            for lanes, ba in forward_pairs(pj, fb, lanes_per_ray, bundles):
                apply_shape(pj, {"shape": (fb, *base_tile), "bundle": ba, "lanes": lanes})
                work.copy_(recon)
                pj.reconstruct(alg, 1, sino, work, params)  # allocation, warm caches
                pj.phase_times(reset=True)
                work.copy_(recon)
                pj.reconstruct(alg, 1, sino, work, params)
                fwd_ms[(fb, lanes, ba)] = pj.phase_times(reset=True)["forward"][0]
                if verbose:
                    print(f"[autotune] forward batch {fb} lanes {lanes} bundle {ba}: "
                          f"{fwd_ms[(fb, lanes, ba)]:.2f} ms", flush=True)
        best_fb, best_lanes, best_ba = min(fwd_ms, key=fwd_ms.get)
        apply_shape(pj, {"shape": (best_fb, *base_tile), "bundle": best_ba, "lanes": best_lanes})
        for t in tiles:
            if t[2] not in tile_batches:
                continue
            for rest in ((False, True) if t[2] == 32 and has_rest(pj.S) else (False,)):
                apply_shape(pj, {"shape": (best_fb, *t), "bundle": best_ba, "lanes": best_lanes,
                                 "rest": rest})
                work.copy_(recon)
                pj.reconstruct(alg, 1, sino, work, params)
                back_ms[(t, rest)] = pj.phase_times(reset=True)["back"][0]
                if verbose:
                    print(f"[autotune] tile {t}{' + rest' if rest else ''}: "
                          f"{back_ms[(t, rest)]:.2f} ms", flush=True)
        best_tile, rest = min(back_ms, key=back_ms.get)
        # no difference for this stack, but for another depth the shape is used at
        rest = rest or not has_rest(pj.S)
    finally:
        pj.set_phase_timing(False)
        torch.cuda.synchronize(pj.device)
    shape = (best_fb, *best_tile)
    res = {"shape": list(shape), "bundle": best_ba, "lanes": best_lanes, "rest": rest,
           "forward_ms": {f"{k[0]}x{k[1]}x{k[2]}": v for k, v in fwd_ms.items()},
           "back_ms": {"x".join(map(str, k)) + ("+rest" if r else ""): v
                       for (k, r), v in back_ms.items()}}
    apply_shape(pj, res)
    _CACHE[key] = res
    if cache_file:
        try:
            with open(cache_file, "w") as f:
                json.dump(_CACHE, f, indent=1)
        except OSError:
            pass
    return res
