// staged.hip -- forward projector with the image staged in LDS, for slice
// batches (a pixel's slices contiguous in xb).
//
// The whole-ray form (kernels.hip) reads every segment's pixel line from
// L2; rays share lines only when they happen to meet in time, so each line
// comes from memory hundreds of times per launch.  Here one workgroup holds
// a bundle of up to kStG angles x kStW adjacent columns (one wavefront per
// angle, one lane per ray) and walks all of its rays together through the
// image in thin slabs across the walk direction:
//
//   * shallow rays (|slope| <= 1) sweep slabs of H pixel columns left to
//     right (the walk is sorted by x, so the pixel column never decreases);
//   * steep rays sweep slabs of H pixel rows, upwards or downwards with the
//     sign of the slope.
//
// A bundle's angles come from the projections sorted by direction, never
// across a change of sweep: a ray swept against its direction would read
// everything from HBM (one such bundle, at 90 degrees, took 34 ms by itself
// where the other bundles of a 1024^2, 720-angle launch take 4), and
// projections need not be given in the order of their angles.
//
// For each slab the workgroup stages the pixels its rays cross (a window
// planned once per geometry from the bundle's outermost rays) in LDS,
// double-buffered, while the lanes consume the previous slab.  Each lane
// still walks its own ray from start to end in the reference's order and
// adds x[idx]*len per slice exactly as the whole-ray form does
// (sirt.cc:4-19), so y is bit-identical; a segment whose pixel is not in the
// staged window (outside the plan's margin, a row wrap at ix == N, a window
// clipped to the buffer) reads its line from HBM instead.  The staging plan
// therefore affects only speed, never the sums.
//
// Bound by vector issue (0.9 of the rate) with the LDS reads close behind: 45
// instructions of walk and window test a segment, a multiply and an add per
// slice.  64 slices of 2048^2 at 1500 angles take 49 ms; 64 with the bundles
// in projection order and the walk before it lost its integer lines, 100 in
// the whole-ray form.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <numeric>

#include "staged.h"

#pragma clang fp contract(off)

namespace trace_hip {

namespace {

// Four floats as a native vector: staged values live in registers across
// the slab loop (an array of the float4 class does not reliably).
typedef float f4 __attribute__((ext_vector_type(4)));
constexpr int kBlock = kStG * 64;  // one wavefront per angle
static_assert(kStW == 64, "one lane per column of the bundle");

// LDS layout and staging order of one slice batch and slab thickness.
template <int SB, int H>
struct Slab {
  static constexpr int kGroups = SB / 4;  // float4 groups of a pixel's slices
  // A pixel's slices take one float4 slot more than they fill (an odd count):
  // the lines of neighbouring pixels then start 4 banks apart, so the lanes
  // of a wavefront reading one group of neighbouring pixels hit different
  // banks, and the groups of a line sit at fixed offsets from its start.
  static constexpr int kPix4 = kGroups == 1 ? 1 : kGroups + 1;
  static constexpr int kE = staged_pixels(SB) / H;  // pixels across a slab
  static constexpr int kRow4 = kE * kPix4;          // slots of one pixel line along the slab
  static constexpr int kBuf4 = H * kRow4;           // slots per buffer
  static constexpr size_t kLds = 2 * (size_t)kBuf4 * sizeof(f4);
  // Thread t stages group t % kGroups of the pixels (du, dv0 + j * kStep)
  static constexpr int kStep = kBlock / kGroups / H;
  static constexpr int kStage = (kE + kStep - 1) / kStep;  // float4 staged per thread
  static_assert(kBlock % (kGroups * H) == 0, "whole pixels per staging pass");
  static_assert(kLds <= 160 * 1024, "two slab buffers must fit the 160 KB of LDS");
};

// Plan of one bundle: per slab the first pixel and the extent of the window
// across the slab (extent 0: nothing to stage).  One block per bundle; the
// window of slab k holds the pixels, with one pixel of margin, that the
// lines of the bundle's outermost rays (first and last column of every
// angle: at a fixed position along the sweep the rays of an angle are
// parallel lines ordered by column) cross within the slab.
__global__ void __launch_bounds__(256)
k_staged_plan(GridInfo g, const RayInfo *__restrict__ rays, const int *__restrict__ order,
              const int4 *__restrict__ group, int H, int emax, int nslab, int ngc,
              int2 *__restrict__ range) {
  const int wg = blockIdx.x;
  const int4 ga = group[wg / ngc];
  const int c0 = (wg % ngc) * kStW;
  const int cn = min(kStW, g.C - c0);
  const int N = g.N, axis = ga.z;
  const double mg = 0.5 * N;
  for (int k = threadIdx.x; k < nslab; k += blockDim.x) {
    // grid-coordinate interval of the slab along the sweep, half a pixel of
    // margin on either side
    const int u0 = (axis == kStAxisYDown ? nslab - 1 - k : k) * H;
    const double ua = (double)u0 - mg - 0.5, ub = (double)(u0 + H) - mg + 0.5;
    double lo = 1e30, hi = -1e30;
    bool any = false, wide = false;
    for (int e = 0; e < 2 * ga.y; ++e) {
      const int p = order[ga.x + (e >> 1)];
      const int c = (e & 1) ? c0 + cn - 1 : c0;
      const RayInfo r = rays[(int64_t)p * g.C + c];
      double va, vb;
      if (axis == kStAxisX) {  // y on the ray at x = ua, ub
        va = (double)r.slope * (ua - (double)r.srcx) + (double)r.srcy;
        vb = (double)r.slope * (ub - (double)r.srcx) + (double)r.srcy;
      } else {                 // x on the ray at y = ua, ub
        va = (double)r.islope * (ua - (double)r.srcy) + (double)r.srcx;
        vb = (double)r.islope * (ub - (double)r.srcy) + (double)r.srcx;
      }
      if (!std::isfinite(va) || !std::isfinite(vb)) {
        wide = true;
        continue;
      }
      lo = fmin(lo, fmin(va, vb));
      hi = fmax(hi, fmax(va, vb));
      any = true;
    }
    int first = 0, last = -1;
    if (wide) {
      first = 0;
      last = N - 1;
    } else if (any) {
      const double fl = floor(lo + mg) - 1.0, fh = floor(hi + mg) + 1.0;
      first = (int)fmax(fl, 0.0);
      last = (int)fmin(fh, (double)(N - 1));
    }
    int extent = last >= first ? last - first + 1 : 0;
    if (extent > emax) {  // keep the middle of the window
      first += (extent - emax) / 2;
      extent = emax;
    }
    range[(int64_t)wg * nslab + k] = make_int2(first, extent);
  }
}

// The walk of one lane, one segment ahead: the pending segment is computed
// but not yet added.
constexpr int kStDone = 1 << 30;  // u of a finished walk, past every slab
template <int AXIS>
struct StagedWalk {
  Walker w;
  float px, py;
  float len, len2;
  int u, v;  // pixel along and across the sweep (a row for u downwards)

  template <bool kExact>
  __device__ __forceinline__ void advance(const GridInfo &g) {
    float qx, qy;
    uint64_t none;
    w.next(qx, qy, none);
    int ix, iy;
    segment<kExact>(px, py, qx, qy, g.mg, ix, iy, len, len2);
    px = qx;
    py = qy;
    u = AXIS == kStAxisX ? ix : iy;
    v = AXIS == kStAxisX ? iy : ix;
    u = __builtin_amdgcn_inverse_ballot_w64(none) ? (AXIS == kStAxisYDown ? -kStDone : kStDone) : u;
  }
};

template <int SB, int H, int MODE, bool kExact, int AXIS>
__device__ __forceinline__ void forward_staged(
    f4 *slab, const int4 &ga, const int *__restrict__ order, int cb, int b, const GridInfo &g,
    const AngleInfo *__restrict__ ang, const RayInfo *__restrict__ rays, int S, int nslab,
    const int2 *__restrict__ rng, const float *__restrict__ xb, const float *__restrict__ sino,
    float *__restrict__ out, unsigned *__restrict__ maxw) {
  using L = Slab<SB, H>;
  const int lane = threadIdx.x & 63;
  const int slot = threadIdx.x >> 6;
  const int p = order[ga.x + min(slot, ga.y - 1)], c = cb * kStW + lane;
  const int C = g.C, N = g.N;
  const bool valid = slot < ga.y && c < C;
  const unsigned NN = (unsigned)N * (unsigned)N;
  const float *xbb = xb + (int64_t)b * NN * SB;

  float acc[SB];
#pragma unroll
  for (int s = 0; s < SB; ++s) acc[s] = 0.f;
  float a2 = 0.f;
  bool hit = false;  // the ray has a segment in the image

  StagedWalk<AXIS> r;
  r.u = AXIS == kStAxisYDown ? -kStDone : kStDone;
  r.v = 0;
  r.len = r.len2 = 0.f;
  const int64_t t = (int64_t)p * C + c;
  if (valid) {
    const RayInfo ri = rays[t];
    hit = (ri.alo & kRayHits) != 0;
    r.w.init(ri, N, ang[p].quadrant);
    r.w.seek(0, 0);
    if (r.w.alen + r.w.blen >= 2) {
      r.w.next(r.px, r.py);
      r.template advance<kExact>(g);
    }
  }

  // this thread's share of a slab: offsets of its pixels in xb from the
  // slab window's first one, and in a buffer
  const int sg = threadIdx.x % L::kGroups, sq = threadIdx.x / L::kGroups;
  const int du = sq % H, dv0 = sq / H;
  const unsigned vstep = (unsigned)(L::kStep * SB * 4) * (AXIS == kStAxisX ? (unsigned)N : 1u);
  const unsigned voff = ((unsigned)(AXIS == kStAxisX ? dv0 : du) * (unsigned)N +
                         (unsigned)(AXIS == kStAxisX ? du : dv0)) * (unsigned)(SB * 4) + 16u * sg;
  const int doff = du * L::kRow4 + dv0 * L::kPix4 + sg;
  f4 stg[L::kStage];
  auto slab_u = [&](int k) { return (AXIS == kStAxisYDown ? nslab - 1 - k : k) * H; };
  auto window = [&](int k, int lo) {  // first pixel of the slab's window in xb
    const int64_t u = slab_u(k);
    return reinterpret_cast<const char *>(
        xbb + (AXIS == kStAxisX ? (int64_t)lo * N + u : u * N + lo) * SB);
  };
  int2 cur = rng[0];
  {
    const char *src = window(0, cur.x);
    const int live = slab_u(0) + du < N ? cur.y : 0;
#pragma unroll
    for (int j = 0; j < L::kStage; ++j)
      if (dv0 + j * L::kStep < live)
        slab[doff + j * (L::kStep * L::kPix4)] =
            *reinterpret_cast<const f4 *>(src + (voff + j * vstep));
  }
  __syncthreads();
  // Slab k: stage slab k + 1 into the other buffer while the lanes add their
  // segments up to slab k (and those of earlier slabs, from HBM: they were
  // not staged).  The pass k == nslab, past the last slab, adds what is left,
  // from HBM (nothing for a ray inside the grid).
  for (int k = 0; k <= nslab; ++k) {
    const bool more = k + 1 < nslab;
    const int2 nxt = more ? rng[k + 1] : make_int2(0, 0);
    const int live = more && slab_u(k + 1) + du < N ? nxt.y : 0;
    if (more) {
      const char *src = window(k + 1, nxt.x);
#pragma unroll
      for (int j = 0; j < L::kStage; ++j)
        if (dv0 + j * L::kStep < live)
          stg[j] = *reinterpret_cast<const f4 *>(src + (voff + j * vstep));
    }
    const bool last = k == nslab;
    // pixels [u0, u1) along the sweep are staged; those the walk has passed
    // or reached are taken (downwards: from u0 on; else: below u1)
    const int u0 = last ? (AXIS == kStAxisYDown ? -1 : N) : slab_u(k);
    const int u1 = last ? (AXIS == kStAxisYDown ? 0 : kStDone) : min(u0 + H, N);
    const int lo = cur.x;
    const unsigned E = last ? 0u : (unsigned)cur.y;
    // byte offset of staged pixel (u, dv) is u * row + dv * pix + base
    const int base = ((k & 1) * L::kBuf4 - u0 * L::kRow4) * 16;
    while (AXIS == kStAxisYDown ? r.u >= u0 : r.u < u1) {
      const unsigned dv = (unsigned)(r.v - lo);
      const bool in_slab = AXIS == kStAxisYDown ? r.u < u1 : r.u >= u0;
      if (in_slab && dv < E) {
        const unsigned lq = __umul24((unsigned)r.u, L::kRow4 * 16) +
                            (__umul24(dv, L::kPix4 * 16) + (unsigned)base);
        const f4 *src = reinterpret_cast<const f4 *>(reinterpret_cast<const char *>(slab) + lq);
        // a quarter to half of the line at a time, so that at most 16 loaded
        // values are live
#pragma unroll
        for (int h = 0; h < L::kGroups; h += 4) {
          f4 f[4];
#pragma unroll
          for (int j = 0; j < 4 && j < L::kGroups; ++j) f[j] = src[h + j];
#pragma unroll
          for (int j = 0; j < 4 && j < L::kGroups; ++j) {
            float *a = acc + 4 * (h + j);
            a[0] += f[j].x * r.len; a[1] += f[j].y * r.len;
            a[2] += f[j].z * r.len; a[3] += f[j].w * r.len;
          }
        }
      } else {
        const unsigned idx = AXIS == kStAxisX ? (unsigned)(r.u + r.v * N) : (unsigned)(r.v + r.u * N);
        if (idx < NN) {
          // from HBM; the explicit wait keeps the merge point free of
          // waits, which would otherwise also wait for the staging loads
          const f4 *gsrc = reinterpret_cast<const f4 *>(xbb + (int64_t)idx * SB);
#pragma unroll
          for (int h = 0; h < L::kGroups; h += 4) {
            f4 f[4];
#pragma unroll
            for (int j = 0; j < 4 && j < L::kGroups; ++j) f[j] = gsrc[h + j];
            wait_vector_loads();
#pragma unroll
            for (int j = 0; j < 4 && j < L::kGroups; ++j) {
              float *a = acc + 4 * (h + j);
              a[0] += f[j].x * r.len; a[1] += f[j].y * r.len;
              a[2] += f[j].z * r.len; a[3] += f[j].w * r.len;
            }
          }
        }
      }
      if (MODE == kFwdOutSIRT) a2 += r.len2;
      r.template advance<kExact>(g);
    }
    if (more) {
      f4 *dst = slab + doff + ((k + 1) & 1) * L::kBuf4;
#pragma unroll
      for (int j = 0; j < L::kStage; ++j)
        if (dv0 + j * L::kStep < live) dst[j * (L::kStep * L::kPix4)] = stg[j];
    }
    // every staging load has been waited for by its store; saying so here
    // keeps the compiler from waiting again before the next slab's loads
    wait_vector_loads();
    if (k < nslab) __syncthreads();
    cur = nxt;
  }

  // the staged pixels are done with: the first words hold the slices' maxima
  unsigned *s_max = reinterpret_cast<unsigned *>(slab);
  if (MODE != kFwdOutY) {
    if (threadIdx.x < SB) s_max[threadIdx.x] = 0;
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < SB; ++k) {
    const int s = b * SB + k;
    const bool live = valid && (s < S);
    unsigned m = 0;
    if (live) {
      const int64_t o = ((int64_t)p * S + s) * C + c;
      if (MODE == kFwdOutY) {
        out[o] = acc[k];
      } else {
        const float wv = (MODE == kFwdOutSIRT) ? (sino[o] - acc[k]) / a2 : sino[o] / acc[k];
        out[t * S + s] = wv;
        // a ray with no segment in the image does not set the scale (as in
        // the whole-ray form)
        if (hit) m = __float_as_uint(__builtin_fabsf(wv));
      }
    }
    if (MODE != kFwdOutY) {
      for (int off = 32; off >= 1; off >>= 1)
        m = max(m, (unsigned)__shfl_down((int)m, off, 64));
      if (lane == 0) atomicMax(s_max + k, m);
    }
  }
  if (MODE != kFwdOutY) {
    __syncthreads();
    const int s = b * SB + threadIdx.x;
    if (threadIdx.x < SB && s < S) raise_max(maxw + s, s_max[threadIdx.x]);
  }
}

template <int SB, int H, int MODE, bool kExact>
__global__ void __launch_bounds__(kBlock)
k_forward_staged(GridInfo g, const AngleInfo *__restrict__ ang,
                 const RayInfo *__restrict__ rays, int S, int nslab, int ngc,
                 const int *__restrict__ order, const int4 *__restrict__ group,
                 const int2 *__restrict__ range, const float *__restrict__ xb,
                 const float *__restrict__ sino, float *__restrict__ out,
                 unsigned *__restrict__ maxw) {
  extern __shared__ f4 slab[];  // [2][Slab::kBuf4]
  const int wg = (int)xcd_chunked(blockIdx.x, gridDim.x);
  const int b = blockIdx.y;
  const int4 ga = group[wg / ngc];
  const int cb = wg % ngc;
  const int2 *rng = range + (int64_t)wg * nslab;
  // uniform: one specialised body per sweep axis
  if (ga.z == kStAxisX)
    forward_staged<SB, H, MODE, kExact, kStAxisX>(slab, ga, order, cb, b, g, ang, rays, S, nslab,
                                                  rng, xb, sino, out, maxw);
  else if (ga.z == kStAxisYUp)
    forward_staged<SB, H, MODE, kExact, kStAxisYUp>(slab, ga, order, cb, b, g, ang, rays, S,
                                                    nslab, rng, xb, sino, out, maxw);
  else
    forward_staged<SB, H, MODE, kExact, kStAxisYDown>(slab, ga, order, cb, b, g, ang, rays, S,
                                                      nslab, rng, xb, sino, out, maxw);
}

template <int SB, int H, int MODE, bool E>
hipError_t staged_launch(const Geometry &g, const RayInfo *rays, const StagedPlan &pl,
                         const float *xb, const float *sino, float *out, unsigned *maxw,
                         hipStream_t st) {
  auto kern = k_forward_staged<SB, H, MODE, E>;
  constexpr size_t lds = Slab<SB, H>::kLds;
  hipError_t e = hipFuncSetAttribute((const void *)kern,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  dim3 grid((unsigned)(pl.ngc * pl.ngroups), (g.S + SB - 1) / SB), block(kBlock);
  hipLaunchKernelGGL(kern, grid, block, lds, st, g.grid, g.d_ang, rays, g.S, pl.nslab, pl.ngc,
                     pl.order, pl.group, pl.range, xb, sino, out, maxw);
  return hipGetLastError();
}

template <int SB, int H>
hipError_t staged_mode(const Geometry &g, const RayInfo *rays, const StagedPlan &pl, int mode,
                       bool exact, const float *xb, const float *sino, float *out,
                       unsigned *maxw, hipStream_t st) {
  if (mode == kFwdOutY)
    return exact ? staged_launch<SB, H, kFwdOutY, true>(g, rays, pl, xb, sino, out, maxw, st)
                 : staged_launch<SB, H, kFwdOutY, false>(g, rays, pl, xb, sino, out, maxw, st);
  if (mode == kFwdOutSIRT)
    return exact ? staged_launch<SB, H, kFwdOutSIRT, true>(g, rays, pl, xb, sino, out, maxw, st)
                 : staged_launch<SB, H, kFwdOutSIRT, false>(g, rays, pl, xb, sino, out, maxw, st);
  return exact ? staged_launch<SB, H, kFwdOutEM, true>(g, rays, pl, xb, sino, out, maxw, st)
               : staged_launch<SB, H, kFwdOutEM, false>(g, rays, pl, xb, sino, out, maxw, st);
}

}  // namespace

StagedLayout staged_layout(const Geometry &g, const AngleInfo *ang, int sb) {
  // Directions from -45 degrees on: shallow, upwards and downwards rays in
  // turn, then the same again pointing the other way (whose columns lie in
  // reverse on the image), each by angle.
  struct Dir {
    double a, t, width;  // direction, its tangent against the sweep, pixels of a column block
    int axis;
    bool reverse;
  };
  std::vector<Dir> dir(g.P);
  for (int p = 0; p < g.P; ++p) {
    const double s = ang[p].sinq, c = ang[p].cosq;
    Dir &d = dir[p];
    d.axis = std::fabs(s) <= std::fabs(c) ? kStAxisX : (s * c > 0 ? kStAxisYUp : kStAxisYDown);
    d.t = d.axis == kStAxisX ? s / c : c / s;
    d.width = kStW / std::max(std::fabs(s), std::fabs(c));
    d.reverse = (d.axis == kStAxisX ? c : s) < 0;
    d.a = std::atan2(s, c) + (std::atan2(s, c) < -M_PI / 4 ? 2 * M_PI : 0.0);
  }
  StagedLayout best;
  std::vector<int> order(g.P);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(),
                   [&](int i, int j) { return dir[i].a < dir[j].a; });
  best.order = order;
  double best_cost = 0;
  // A group takes angles while its window stays within the buffer's at the
  // image's edge; where the bundles fill the GPU at least twice over, within
  // a quarter more (clipped there, where few rays are: a clipped slab waits
  // for HBM, which other bundles then hide.  One 32-slice batch, limits 1.25
  // and 1: 24.5 and 26.2 ms at 2048^2 / 1500 angles, 0.83 and 0.69 ms at
  // 512^2 / 360).
  const int64_t bundles =
      (int64_t)((g.P + kStG - 1) / kStG) * ((g.C + kStW - 1) / kStW) * ((g.S + sb - 1) / sb);
  const double over = bundles >= 512 ? 1.25 : 1.0;
  for (int H : {4, 2, 1}) {
    if (H == 1 && sb != 32) continue;
    const double limit = over * staged_pixels(sb) / H;
    std::vector<int4> group;
    double cost = 0;
    for (int i = 0; i < g.P;) {
      const Dir &d0 = dir[order[i]];
      int n = 1;
      while (i + n < g.P && n < kStG) {
        const Dir &d = dir[order[i + n]];
        if (d.axis != d0.axis || d.reverse != d0.reverse) break;
        const double e = std::max(d0.width, d.width) + 0.5 * g.N * std::fabs(d.t - d0.t) + 4.0;
        if (e > limit) break;
        ++n;
      }
      group.push_back(make_int4(i, n, d0.axis, 0));
      cost += std::max(n, kStG / 2) * 1.4 * (45.0 + 2 * sb) + kStG * 60.0 / H;
      i += n;
    }
    if (best.H == 0 || cost < best_cost) {
      best.H = H;
      best.group = group;
      best_cost = cost;
    }
  }
  // Each XCD runs a contiguous eighth of the workgroups (xcd_chunked).  A
  // diagonal bundle takes up to 2.8 times as long as one along an axis, so
  // the groups are dealt to the eighths in turn, longest first.
  auto length = [&](const int4 &ga) {
    const Dir &d = dir[order[ga.x + ga.y / 2]];
    return d.width * ga.y;
  };
  std::stable_sort(best.group.begin(), best.group.end(),
                   [&](const int4 &i, const int4 &j) { return length(i) > length(j); });
  std::vector<int4> dealt;
  for (size_t x = 0; x < 8; ++x)
    for (size_t i = x; i < best.group.size(); i += 8) dealt.push_back(best.group[i]);
  best.group = dealt;
  return best;
}

// A staged launch sweeps every bundle through the image however few its rays
// are, which takes 0.5 to 1 us a pixel of the side; the other forms take their
// segments' gathers, which cost the more the further the image outgrows the
// caches and the fewer the angles whose rays could share lines.  The side to the
// power 1.75 times the angles tells the faster form, with a least number of
// angles (bundles of few angles sweep for few rays) and, at 4 and 8 slices, a
// least side (smaller images stay in the L2s).  Over 277 geometries a batch, N
// from 128 to 2048 and 30 to 1500 uniform angles, the choice lies above the
// better form by 0.3, 0.7, 1.0 and 0.9% on average at 4, 8, 16 and 32 slices, and
// by more than 10% in 4, 6, 11 and 10 of them (by 43% at most; what remains is the
// grouping's steps, as between 1300^2 and 1600^2 below).  Staged / the better of
// the others (us):
//                4 slices      8 slices     16 slices      32 slices
//   256^2, 1500    228 / 251     257 / 236     379 / 437     518 / 535
//   512^2,  500    359 / 347     396 / 431     498 / 683     977 / 838
//   600^2, 1000    736 / 708     826 / 777    1343 / 1487   1880 / 2131
//   725^2,  720    826 / 600     904 / 975    1461 / 1726   1987 / 2462
//   900^2,  130    604 / 362     520 / 506     682 / 764    1152 / 1434
//   900^2,  250    617 / 683     880 / 857     867 / 1303   1513 / 1747
//  1100^2,   90    662 / 377     883 / 623    1119 / 933    1212 / 1763
//  1300^2,   60    998 / 368     875 / 592    1197 / 900    2038 / 1896
//  1300^2,  250   1116 / 1474   1171 / 1953   2170 / 2839   3317 / 5445
//  1600^2,   60   1224 / 535    1439 / 923    1350 / 1509   2296 / 2962
//  2048^2,   60   1565 / 810    1665 / 1408   3396 / 2292   5244 / 5010
//  2048^2,  130   1707 / 2691   2076 / 3001   3910 / 4851   6832 / 11707
// Projections in no order of direction (random or shuffled angles) leave the other
// forms' bundles of adjacent projections nothing to share, and the staged form,
// which sorts them, wins from fewer rays on: 100 geometries a batch, 0 to 0.8%
// above the better form on average.  Staged / others (us) at random angles:
// 4 slices 822^2, 908 angles 1219 / 2335; 8 slices 600^2, 400 631 / 732; 32 slices
// 300^2, 400 443 / 394.
bool staged_faster(const Geometry &g, int sb, bool scattered) {
  const double side = std::min(g.N, g.C), root = std::sqrt(side);
  struct Limit {
    int side, angles;
    double work;
  };
  if (scattered) {
    const Limit l = sb == 4    ? Limit{450, 0, 1.97e5}
                    : sb == 8  ? Limit{330, 0, 1.52e5}
                    : sb == 16 ? Limit{256, 0, 1.02e5}
                               : Limit{256, 0, 8.9e4};
    return side >= l.side && side * g.P >= l.work;
  }
  const Limit l = sb == 4    ? Limit{950, 100, 4.5e7}
                  : sb == 8  ? Limit{512, 90, 3.75e7}
                  : sb == 16 ? Limit{0, 70, 1.6e7}
                             : Limit{0, 60, 1.84e7};
  return side >= l.side && g.P >= l.angles && side * root * std::sqrt(root) * g.P >= l.work;
}

// Successive projections turned against each other by more than a quarter radian
// on average (two directions at random: 2/pi in the sine; P over a half turn: pi/P).
bool scattered_angles(const AngleInfo *ang, int P) {
  double turn = 0;
  for (int p = 1; p < P; ++p)
    turn += std::fabs((double)ang[p].sinq * ang[p - 1].cosq - (double)ang[p].cosq * ang[p - 1].sinq);
  return P > 1 && turn > 0.25 * (P - 1);
}

hipError_t launch_staged_plan(const Geometry &g, const RayInfo *rays, StagedPlan &pl,
                              hipStream_t st) {
  hipLaunchKernelGGL(k_staged_plan, dim3(pl.ngroups * pl.ngc), dim3(256), 0, st, g.grid, rays,
                     pl.order, pl.group, pl.H, staged_pixels(pl.sb) / pl.H, pl.nslab, pl.ngc,
                     pl.range);
  return hipGetLastError();
}

hipError_t launch_forward_staged(const Geometry &g, const RayInfo *rays, const StagedPlan &pl,
                                 int mode, bool exact, const float *xb, const float *sino,
                                 float *out, unsigned *maxw, hipStream_t st) {
#define TRACE_ST_CASE(SB_, H_)                                                             \
  if (pl.sb == SB_ && pl.H == H_)                                                          \
    return staged_mode<SB_, H_>(g, rays, pl, mode, exact, xb, sino, out, maxw, st);
  TRACE_ST_CASE(32, 4)
  TRACE_ST_CASE(32, 2)
  TRACE_ST_CASE(32, 1)
  TRACE_ST_CASE(16, 4)
  TRACE_ST_CASE(16, 2)
  TRACE_ST_CASE(8, 4)
  TRACE_ST_CASE(8, 2)
  TRACE_ST_CASE(4, 4)
  TRACE_ST_CASE(4, 2)
#undef TRACE_ST_CASE
  return hipErrorInvalidValue;
}

}  // namespace trace_hip
