// split.hip -- forward projector for launches of few rays.
//
// The whole-ray form (kernels.hip) walks a ray with one lane from end to end,
// since its sum must be added up in the reference's order.  A small launch has
// fewer wavefronts than the GPU has SIMDs, and its time is that of the longest
// walk: some 300 clocks a segment.  Only the additions need the order.  Here K
// lanes share a ray: each walks every K-th piece of kPiece segments, gathers,
// and leaves the products x * len in LDS; then one lane per (ray, slice) adds
// the products of the K pieces one after the other, exactly as the whole walk
// does (sirt.cc:4-19).  The sums are therefore bit-identical.
//
// A piece starts at a merged point known only by its number: the state of the
// merge after k points is found by bisection over the A list (merge_seek),
// exact because the lists are sorted.  A ray whose A list is not ascending in
// walk order (angles below -pi/2) has no such state; its first lane then walks
// all the pieces.
//
// Bound by vector issue from some 50 thousand rays on, below by the walk of
// one lane's pieces.  256^2 at 180 angles: 56 -> 35 us a launch; the rule of
// split_lanes holds both sides.
#include <hip/hip_runtime.h>

#include "internal.h"

#pragma clang fp contract(off)

namespace trace_hip {

namespace {

constexpr int kBlock = 128;

// State of the merge after k points, 0 <= k <= alen + blen: the walker's heads
// become element i of A and j = k - i of B.  i is the smallest number of A
// elements for which A[i] does not come before B[k - i - 1]: A wins only on a
// strict less-than (Walker::next).
__device__ __forceinline__ void merge_seek(Walker &w, int k) {
  int lo = max(0, k - w.blen), hi = min(k, w.alen);
  while (lo < hi) {
    const int m = (lo + hi) >> 1;  // A[m] exists: m < hi <= alen; B[k - m - 1]: m < k
    if (w.cross_a(w.a_line(m)) < grid_line(w.N, w.blo + k - m - 1)) lo = m + 1;
    else hi = m;
  }
  w.seek(lo, k - lo);
}

// LDS of one wavefront: products [ray][segment of the round][slice], and for
// the squared lengths [ray][segment].
template <int SB, int K, int M>
struct SplitLds {
  static constexpr int kRays = 64 / K;
  static constexpr int kChunk = M * SB + 4;       // floats of a piece, padded
  static constexpr int kRay = K * kChunk + 4;     // floats of a ray's pieces, padded
  float prod[kRays * kRay];
};

template <int SB, int K, int M, int MODE, bool kExact>
__global__ void __launch_bounds__(kBlock)
k_forward_split(GridInfo g, const AngleInfo *__restrict__ ang, const RayInfo *__restrict__ rays,
                int P, int S, int xsb, const float *__restrict__ xb,
                const float *__restrict__ sino, float *__restrict__ out,
                unsigned *__restrict__ maxw) {
  using L = SplitLds<SB, K, M>;
  using L2 = SplitLds<1, K, M>;
  constexpr bool kSq = MODE == kFwdOutSIRT;
  constexpr int R = L::kRays;
  constexpr int U = SB == 1 ? 8 : 4;  // gathers in flight
  static_assert(M % U == 0, "whole sets of gathers");
  __shared__ __align__(16) float s_prod[kBlock / 64][L::kRays * L::kRay];
  __shared__ __align__(16) float s_sq[kSq ? kBlock / 64 : 1][kSq ? L2::kRays * L2::kRay : 1];
  __shared__ unsigned s_max[SB];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int sub = lane / R, r = lane % R;
  const int C = g.C, N = g.N;
  const int64_t nrays = (int64_t)P * C;
  const int64_t first =
      ((int64_t)xcd_chunked(blockIdx.x, gridDim.x) * (kBlock / 64) + wv) * R;  // of this wavefront
  const int sbase = blockIdx.y * SB;
  if (MODE != kFwdOutY) {
    if (threadIdx.x < SB) s_max[threadIdx.x] = 0;
    __syncthreads();
  }
  float *prod = s_prod[wv] + r * L::kRay;
  float *sq = kSq ? s_sq[wv] + r * L2::kRay : nullptr;

  const bool valid = first + r < nrays;
  const int64_t t = valid ? first + r : 0;
  Walker w;
  w.init(rays[t], N, ang[t / C].quadrant);
  w.seek(0, 0);
  const int nseg = valid ? max(0, w.alen + w.blen - 1) : 0;
  const bool sorted = w.a_sorted();
  const bool any_whole = __any(nseg > 0 && !sorted) != 0;
  int most = nseg;
  for (int off = 32; off > 0; off >>= 1) most = max(most, __shfl_xor(most, off, 64));
  const int most_u = __builtin_amdgcn_readfirstlane(most);

  const unsigned bytes = (unsigned)N * (unsigned)N * (unsigned)(xsb * 4);
  const float *xp = xb + (int64_t)(sbase / xsb) * N * N * xsb;
  const auto rsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(xp), 0, (int)bytes, 0x00027000);
  const unsigned skip = (unsigned)(sbase % xsb) * 4, stride = (unsigned)(xsb * 4);

  // this lane's sums: (slice or squared length, ray) items of the wavefront
  constexpr int kItems = R * (SB + (kSq ? 1 : 0));
  constexpr int kOwn = (kItems + 63) / 64;
  float acc[kOwn];
#pragma unroll
  for (int i = 0; i < kOwn; ++i) acc[i] = 0.f;

  float px = 0.f, py = 0.f;
  for (int base = 0; base < most_u; base += K * M) {
    // this lane's piece of the round: cnt segments from k0 on
    const int k0 = sorted ? base + sub * M : base;
    const int room = sorted ? M : (sub == 0 ? K * M : 0);
    const int cnt = max(0, min(room, nseg - k0));
    if (cnt > 0 && (sorted || base == 0)) {
      if (sorted) merge_seek(w, k0);
      w.next(px, py);
    }
    const int steps = any_whole ? K * M : M;
    for (int j0 = 0; j0 < steps; j0 += U) {
      float v[U][SB], l[U], l2[U];
      // steps past a lane's count go on from an exhausted walk: their gathers
      // stay inside the resource, or read 0, and their products are not kept
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float qx, qy;
        w.next(qx, qy);
        int ix, iy;
        segment<kExact>(px, py, qx, qy, g.mg, ix, iy, l[u], l2[u]);
        px = qx;
        py = qy;
        const unsigned off = (__umul24(iy, N) + (unsigned)ix) * stride + skip;
        if constexpr (SB == 1) {
          v[u][0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, off, 0, 0));
        } else if constexpr (SB == 2) {
          const auto q = __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, 0, 0);
          v[u][0] = __uint_as_float(q[0]), v[u][1] = __uint_as_float(q[1]);
        } else {
          const auto q = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) v[u][i] = __uint_as_float(q[i]);
        }
      }
      // places past the ray's end hold 0: a sum that starts at +0 keeps its
      // bits when +0 is added
      if (j0 < room) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int j = sub * M + j0 + u;  // place in the round
          const bool go = j0 + u < cnt;
          float *d = prod + (j / M) * L::kChunk + (j % M) * SB;
#pragma unroll
          for (int i = 0; i < SB; ++i) v[u][i] = go ? v[u][i] * l[u] : 0.f;
          if constexpr (SB == 1) d[0] = v[u][0];
          else if constexpr (SB == 2) *reinterpret_cast<float2 *>(d) = make_float2(v[u][0], v[u][1]);
          else *reinterpret_cast<float4 *>(d) = make_float4(v[u][0], v[u][1], v[u][2], v[u][3]);
          if (kSq) sq[(j / M) * L2::kChunk + j % M] = go ? l2[u] : 0.f;
        }
      }
    }
    // one lane per (ray, slice): the round's products in order.  Only this
    // wavefront has written them, and its LDS accesses take effect in order.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
      const int item = lane + 64 * i;
      const int what = item / R, ray = item % R;
      if (item < kItems) {
        if (SB == 1 || (kSq && what == SB)) {
          const float *src = (kSq && what == SB) ? s_sq[wv] + ray * L2::kRay
                                                 : s_prod[wv] + ray * L::kRay;
#pragma unroll
          for (int k = 0; k < K; ++k) {
#pragma unroll
            for (int j = 0; j < M; j += 4) {
              const float4 q = *reinterpret_cast<const float4 *>(src + k * L2::kChunk + j);
              acc[i] += q.x;
              acc[i] += q.y;
              acc[i] += q.z;
              acc[i] += q.w;
            }
          }
        } else {
          const float *src = s_prod[wv] + ray * L::kRay + what;
          for (int k = 0; k < K; ++k) {
#pragma unroll
            for (int j = 0; j < M; ++j) acc[i] += src[k * L::kChunk + j * SB];
          }
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }

#pragma unroll
  for (int i = 0; i < kOwn; ++i) {
    // the ray's sum of squared lengths, held by another lane
    float a2 = 0.f;
    const int item = lane + 64 * i;
    const int what = item / R, ray = item % R;
    if (kSq) a2 = __shfl(acc[SB * R / 64], (SB * R + ray) % 64, 64);
    const int s = sbase + what;
    const int64_t tr = first + ray;
    const bool live = what < SB && tr < nrays && s < S;
    if (live) {
      const int64_t p = tr / C, c = tr - p * C;
      const int64_t o = (p * S + s) * C + c;
      if (MODE == kFwdOutY) {
        out[o] = acc[i];
      } else {
        const float wv2 = kSq ? (sino[o] - acc[i]) / a2 : sino[o] / acc[i];
        out[tr * S + s] = wv2;
        // a ray with no segment in the image does not set the scale (as in
        // the whole-ray form)
        if (rays[tr].alo & kRayHits)
          atomicMax(s_max + what, __float_as_uint(__builtin_fabsf(wv2)));
      }
    }
  }
  if (MODE != kFwdOutY) {
    __syncthreads();
    const int s = sbase + threadIdx.x;
    if (threadIdx.x < SB && s < S) raise_max(maxw + s, s_max[threadIdx.x]);
  }
}

template <int SB, int K, int M, int MODE>
hipError_t split_launch(const Geometry &g, const RayInfo *rays, int xsb, bool exact,
                        const float *xb, const float *sino, float *out, unsigned *maxw,
                        hipStream_t st) {
  const int64_t waves = (g.rays_per_slice() + 64 / K - 1) / (64 / K);
  const dim3 grid((unsigned)((waves + kBlock / 64 - 1) / (kBlock / 64)), (g.S + SB - 1) / SB);
  if (exact)
    hipLaunchKernelGGL((k_forward_split<SB, K, M, MODE, true>), grid, dim3(kBlock), 0, st, g.grid,
                       g.d_ang, rays, g.P, g.S, xsb, xb, sino, out, maxw);
  else
    hipLaunchKernelGGL((k_forward_split<SB, K, M, MODE, false>), grid, dim3(kBlock), 0, st, g.grid,
                       g.d_ang, rays, g.P, g.S, xsb, xb, sino, out, maxw);
  return hipGetLastError();
}

template <int SB, int K, int M>
hipError_t split_mode(const Geometry &g, const RayInfo *rays, int xsb, int mode, bool exact,
                      const float *xb, const float *sino, float *out, unsigned *maxw,
                      hipStream_t st) {
  if (mode == kFwdOutY)
    return split_launch<SB, K, M, kFwdOutY>(g, rays, xsb, exact, xb, sino, out, maxw, st);
  if (mode == kFwdOutSIRT)
    return split_launch<SB, K, M, kFwdOutSIRT>(g, rays, xsb, exact, xb, sino, out, maxw, st);
  return split_launch<SB, K, M, kFwdOutEM>(g, rays, xsb, exact, xb, sino, out, maxw, st);
}

}  // namespace

// The split form takes more instructions a segment (places, LDS, the sums by
// few lanes), so it serves where the whole-ray form leaves the GPU waiting: few
// rays, or, at four slices, images past the L2s, whose gathers it has more of in
// flight.  With 8 slices and more it gathers part of a pixel's line at a time
// and pays for the smallest launches only.  One launch, whole / 4 / 8 lanes (us):
//   1 slice     64^2,  48 angles   15 /   8 /   6    256^2, 180   56 /   43 /  35
//              512^2, 360         202 / 209 / 169   1024^2, 180  428 /  389 / 329
//             1024^2, 720        1178 /1434 /1147
//   2 slices   256^2, 180          58 /  43 /  42   1024^2, 180  597 /  531 / 591
//             1024^2, 720        1531 /2136 /2328
//   4 slices   256^2, 180          64 /  56 /  50    320^2, 256  112 /   96 /  98
//              512^2, 360         261 / 285 / 304   1024^2, 180  778 /  606 / 652
//   8 slices   128^2, 100          34 /  19 /  24    256^2, 180   68 /   88 /  93
//  32 slices    64^2,  48          19 /  15 /  17    128^2, 100   36 /   79 /  99
int split_lanes(const Geometry &g, int sb) {
  if (wide_image(g.N, sb)) return 0;
  const int64_t rays = g.rays_per_slice();
  if (sb == 1) return rays <= 500000 ? 8 : 0;
  if (sb == 2) return rays <= 64000 ? 8 : (rays <= 250000 ? 4 : 0);
  if (sb == 4) {
    const bool past_l2 = (int64_t)g.N * g.N * 16 > (int64_t(8) << 20);
    return rays <= 64000 ? 8 : (rays <= (past_l2 ? 200000 : 100000) ? 4 : 0);
  }
  return rays * sb <= 102400 ? (rays <= 4096 ? 8 : 4) : 0;
}

hipError_t launch_forward_split(const Geometry &g, const RayInfo *rays, int sb, int lanes,
                                int mode, bool exact, const float *xb, const float *sino,
                                float *out, unsigned *maxw, hipStream_t st) {
  if (wide_image(g.N, sb)) return hipErrorInvalidValue;
#define TRACE_SPLIT_CASE(SB_, K_, M_)                                                      \
  if ((sb < 4 ? sb : 4) == SB_ && lanes == K_)                                             \
    return split_mode<SB_, K_, M_>(g, rays, sb, mode, exact, xb, sino, out, maxw, st);
  TRACE_SPLIT_CASE(1, 8, 16)
  TRACE_SPLIT_CASE(2, 4, 16)
  TRACE_SPLIT_CASE(2, 8, 16)
  TRACE_SPLIT_CASE(4, 4, 16)
  TRACE_SPLIT_CASE(4, 8, 16)
#undef TRACE_SPLIT_CASE
  return hipErrorInvalidValue;
}

}  // namespace trace_hip
