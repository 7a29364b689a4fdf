// kernels.hip -- gfx950 kernels of the reconstruction hot path.
//
// Data layout in HBM (per handle):
//   x      [S][N][N]        image, the reference's layout (idx = ix + iy*N)
//   xb     [S/SB][N*N][SB]  slice-batched copy of x read by the forward
//                           projector: one segment gathers SB slices as
//                           contiguous float4s
//   w      [P][S][C]        per-ray weights written by the forward projector
//   z      [S][N][N]        A^T w written by the tile backprojector
//   den    [N][N]           A^T 1 (iteration invariant, one slice's geometry)
//   rays   [P][C]           RayInfo: source point, slopes, trimmed ranges
//
// Forward projector: 1, 2 or 4 lanes per ray (p, c) and slice batch, each
// summing its share of the batch's slices; a wavefront holds a bundle of
// adjacent angles x adjacent detector columns.  Each lane walks the whole
// ray in the reference's order and accumulates y = sum x[idx]*len per
// slice, so y is bit-identical to CalculateSimdata (sirt.cc:4-19).
//
// Backprojector: one workgroup per (image tile, slice batch) owns the tile's
// accumulators in LDS for all angles.  Its lanes take the (angle, column)
// pairs whose ray can touch the tile, walk only the part of the ray near the
// tile (traverse_window) and add the fixed-point terms of len*w into LDS
// with integer atomics; the tile is then written to HBM with coalesced
// stores.  No global atomics, no per-thread image replicas (the reference's
// DISP replicas + tree merge, disp_engine_reduction.h:104-185).
#include <hip/hip_runtime.h>

#include <climits>
#include <type_traits>

#include "internal.h"

#pragma clang fp contract(off)

namespace trace_hip {

namespace {

constexpr int kRayBlock = 256;

constexpr int kPixBlock = 256;
constexpr int kTileBlock = 256;

__device__ __forceinline__ void atomic_add_f32(float *p, float v) {
  unsafeAtomicAdd(p, v);  // hardware global float atomic, relaxed
}

// ---------------------------------------------------------------- rays --

// Ray table.  With `counts` also the rays' flags and the geometry's segment
// statistics, from one walk of each ray: all segments, those outside the image,
// the bits of the longest, the rays with a wrapped one and those walked whole
// by the tile kernels (zeroed beforehand).
// Whole-ray walks (the forward projector) read neither.
__global__ void __launch_bounds__(kRayBlock)
k_ray_info(GridInfo g, const AngleInfo *__restrict__ ang, const float *__restrict__ yi,
           int P, unsigned long long *__restrict__ counts, RayInfo *__restrict__ rays) {
  const int64_t t = (int64_t)blockIdx.x * kRayBlock + threadIdx.x;
  const bool valid = t < (int64_t)P * g.C;
  RayStats st;
  unsigned wraps = 0, whole = 0;
  if (valid) {
    const int c = (int)(t % g.C), p = (int)(t / g.C);
    RayInfo r = make_ray(g, yi[c], ang[p].sinq, ang[p].cosq);
    if (counts) {
      r.alo |= ray_flags(g, r, ang[p].quadrant, st);
      wraps = (r.alo & kRayWraps) ? 1u : 0u;
      whole = st.whole ? 1u : 0u;
    }
    rays[t] = r;
  }
  if (!counts) return;
  __shared__ unsigned s_sum[4], s_longest;
  if (threadIdx.x < 4) s_sum[threadIdx.x] = 0;
  if (threadIdx.x == 4) s_longest = 0;
  __syncthreads();
  unsigned lb = __float_as_uint(st.longest);
  for (int off = 32; off > 0; off >>= 1) {
    st.segments += __shfl_down(st.segments, off, 64);
    st.outside += __shfl_down(st.outside, off, 64);
    wraps += __shfl_down(wraps, off, 64);
    whole += __shfl_down(whole, off, 64);
    lb = max(lb, (unsigned)__shfl_down((int)lb, off, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(s_sum + 0, st.segments);
    atomicAdd(s_sum + 1, st.outside);
    atomicAdd(s_sum + 2, wraps);
    atomicAdd(s_sum + 3, whole);
    atomicMax(&s_longest, lb);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    atomicAdd(counts + 0, (unsigned long long)s_sum[0]);
    if (s_sum[1]) atomicAdd(counts + 1, (unsigned long long)s_sum[1]);
    raise_max(reinterpret_cast<unsigned *>(counts + 2), s_longest);
    if (s_sum[2]) atomicAdd(counts + 3, (unsigned long long)s_sum[2]);
    if (s_sum[3]) atomicAdd(counts + 4, (unsigned long long)s_sum[3]);
  }
}

// ------------------------------------------------------------- forward --

enum FwdMode { kFwdY = 0, kFwdSIRT = 1, kFwdEM = 2 };

template <int SB>
struct Vec {
  float v[SB];
};

template <int SB>
__device__ __forceinline__ void store_slices(float *__restrict__ p, const float (&v)[SB]) {
  if constexpr (SB == 1) {
    p[0] = v[0];
  } else if constexpr (SB == 2) {
    *reinterpret_cast<float2 *>(p) = make_float2(v[0], v[1]);
  } else {
#pragma unroll
    for (int q = 0; q < SB; q += 4)
      *reinterpret_cast<float4 *>(p + q) = make_float4(v[q], v[q + 1], v[q + 2], v[q + 3]);
  }
}

// Lanes are grouped in ray bundles: a wavefront holds BA adjacent angles x
// (64 / BA) adjacent detector columns (runtime `ba`), so at every step its
// lanes sit on nearby pixels of nearby rays and share cache lines.  One lane
// per ray (p, c) and slice batch b (blockIdx.y).  kFwdY writes y[p][s][c];
// kFwdSIRT / kFwdEM write the per-ray weight of UpdateReconReplica
//   SIRT  w = (p - y)/a2, a2 = sum len^2    (sirt.cc:47-52)
//   EM    w = p/y                           (mlem.cc:50, pml.cc:236)
// to w[p][c][s] (slices innermost, read as a block by the backprojector) and
// fold max |w| over the rays with a segment in the image per slice into the
// workgroup's s_max[SB] (LDS, bits; zeroed beforehand).
// LPR lanes per ray (1, 2 or 4): the lanes of one ray repeat its walk and
// each gathers and sums SB/LPR of the batch's slices, so a gather touches
// LPR-fold fewer distinct cache lines per wavefront instruction (the
// address unit, not the VALU, limits the one-lane form).
//
// A lane walks K segments, issuing their gathers as it goes, and adds the
// previous K meanwhile, in the walk's order: one segment's gather at a time
// left a small launch (fewer wavefronts than the GPU holds) waiting for
// memory at every step (one slice: 256^2 at 180 angles 102 -> 60 us a launch,
// 2048^2 at 1500 angles, where full occupancy hides most of it, 8.7 -> 8.1 ms;
// there the L1's line rate is the next bound, one line a clock).
//
// Gathers go through a buffer resource over the slice batch: an index past
// the image (the reference's truncation sends a segment there) is outside
// the resource's range and reads 0, and a sum that starts at +0 keeps its
// bits when +0 is added, so no step tests its index.  kWide is the form for
// images of 2^32 bytes and more, which a resource cannot cover.
template <int SBL, bool kWide>
struct ImageGather {
  const float *base;
  __amdgpu_buffer_rsrc_t rsrc;
  unsigned NN;
  int N, stride;  // stride: floats per pixel
  __device__ __forceinline__ ImageGather(const float *p, int N_, int stride_, int skip)
      : base(p + skip), NN((unsigned)N_ * (unsigned)N_), N(N_), stride(stride_) {
    if constexpr (!kWide)
      rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), 0,
                                               (int)(NN * (unsigned)(stride_ * 4)), 0x00027000);
  }
  __device__ __forceinline__ void load(int ix, int iy, int skip_bytes, float (&o)[SBL]) const {
    if constexpr (kWide) {
      const unsigned idx = (unsigned)(ix + iy * N);
#pragma unroll
      for (int k = 0; k < SBL; ++k) o[k] = idx < NN ? base[(int64_t)idx * stride + k] : 0.f;
    } else {
      // ix, iy lie in [0, N]: the midpoints of points inside the square
      const unsigned off = (__umul24(iy, N) + (unsigned)ix) * (unsigned)(stride * 4) + skip_bytes;
      if constexpr (SBL == 1) {
        o[0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, off, 0, 0));
      } else if constexpr (SBL == 2) {
        const auto q = __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, 0, 0);
        o[0] = __uint_as_float(q[0]); o[1] = __uint_as_float(q[1]);
      } else {
#pragma unroll
        for (int k = 0; k < SBL; k += 4) {
          const auto q = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off + 4 * k, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) o[k + i] = __uint_as_float(q[i]);
        }
      }
    }
  }
};

template <int SB, int MODE, bool kExact, int LPR = 1, bool kWide = false>
__device__ __forceinline__ void forward_bundle(const GridInfo &g, const AngleInfo *__restrict__ ang,
                                               const RayInfo *__restrict__ rays, int P, int S,
                                               int ba_log2, const float *__restrict__ xb,
                                               const float *__restrict__ sino,
                                               float *__restrict__ out, unsigned *s_max,
                                               int64_t bundle, int b) {
  static_assert(LPR == 1 || LPR == 2 || LPR == 4, "lanes per ray: 1, 2 or 4");
  static_assert(SB % LPR == 0, "slice batch must split evenly over the lanes of a ray");
  constexpr int SBL = SB / LPR;  // slices per lane
  constexpr int LPR_LOG2 = LPR == 1 ? 0 : (LPR == 2 ? 1 : 2);
  // segments per set (half of those in flight per lane)
  constexpr int K = SBL <= 2 ? 4 : (SBL <= 8 ? 2 : 1);
  const int C = g.C;
  const int lane = threadIdx.x & 63;
  const int sub = lane & (LPR - 1);    // slice group of this lane
  const int rl = lane >> LPR_LOG2;     // ray of this lane within the wavefront
  const int bc_log2 = 6 - LPR_LOG2 - ba_log2;  // columns per bundle = 64 / (LPR * BA)
  const int nbc = (C + (1 << bc_log2) - 1) >> bc_log2;
  const int p = (int)(bundle / nbc) * (1 << ba_log2) + (rl >> bc_log2);
  const int c = (int)(bundle % nbc) * (1 << bc_log2) + (rl & ((1 << bc_log2) - 1));
  const bool valid = (p < P) && (c < C);
  const int64_t NN = (int64_t)g.N * g.N;
  const ImageGather<SBL, kWide> img(xb + b * NN * SB, g.N, SB, sub * SBL);
  const int skip = sub * SBL * 4;
  float acc[SBL];
#pragma unroll
  for (int k = 0; k < SBL; ++k) acc[k] = 0.f;
  float a2 = 0.f;
  bool hit = false;  // the ray has a segment in the image
  const int64_t t = (int64_t)p * C + c;
  if (valid) {
    const RayInfo r = rays[t];
    hit = (r.alo & kRayHits) != 0;
    Walker w;
    w.init(r, g.N, ang[p].quadrant);
    w.seek(0, 0);
    int rem = w.alen + w.blen - 1;  // segments left
    if (rem >= 1) {
      float px, py;
      w.next(px, py);
      // two sets of K segments, one walked while the other is added
      float v[2 * K][SBL], l[2 * K], l2[2 * K];
#pragma unroll
      for (int u = K; u < 2 * K; ++u) {
        l[u] = l2[u] = 0.f;
#pragma unroll
        for (int k = 0; k < SBL; ++k) v[u][k] = 0.f;
      }
      auto step = [&](int u) {
        float qx, qy;
        w.next(qx, qy);
        int ix, iy;
        segment<kExact>(px, py, qx, qy, g.mg, ix, iy, l[u], l2[u]);
        px = qx;
        py = qy;
        img.load(ix, iy, skip, v[u]);
      };
      auto add = [&](int u) {
#pragma unroll
        for (int k = 0; k < SBL; ++k) acc[k] += v[u][k] * l[u];
        if (MODE == kFwdSIRT) a2 += l2[u];
      };
      // the scheduling barriers keep each set's sums after the other set's
      // gathers: moved up, they would wait for loads just issued
      for (; rem >= 2 * K; rem -= 2 * K) {
#pragma unroll
        for (int u = 0; u < K; ++u) step(u);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = K; u < 2 * K; ++u) add(u);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = K; u < 2 * K; ++u) step(u);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < K; ++u) add(u);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int u = K; u < 2 * K; ++u) add(u);
      // what is left, its gathers again all issued before the first is used
#pragma unroll
      for (int u = 0; u < 2 * K - 1; ++u)
        if (u < rem) step(u);
#pragma unroll
      for (int u = 0; u < 2 * K - 1; ++u)
        if (u < rem) add(u);
    }
  }
#pragma unroll
  for (int k = 0; k < SBL; ++k) {
    const int s = b * SB + sub * SBL + k;
    const bool live = valid && (s < S);
    unsigned m = 0;
    if (live) {
      const int64_t o = ((int64_t)p * S + s) * C + c;
      if (MODE == kFwdY) {
        out[o] = acc[k];
      } else {
        const float wv = (MODE == kFwdSIRT) ? (sino[o] - acc[k]) / a2 : sino[o] / acc[k];
        out[t * S + s] = wv;
        // A ray with no segment in the image (a shifted rotation centre
        // leaves edge columns outside) gets y = 0 and a2 = 0, so an
        // inf/NaN weight, as in the reference; it adds nothing to A^T w
        // there or here, so it must not set the slice's scale either.
        if (hit) m = __float_as_uint(__builtin_fabsf(wv));
      }
    }
    if (MODE != kFwdY) {
      // max over the lanes holding the same slice (same sub)
      for (int off = 32; off >= LPR; off >>= 1)
        m = max(m, (unsigned)__shfl_down((int)m, off, 64));
      if (lane < LPR) atomicMax(s_max + sub * SBL + k, m);
    }
  }
}

template <int SB, int MODE, bool kExact, int LPR, bool kWide = false>
__global__ void __launch_bounds__(kRayBlock)
k_forward(GridInfo g, const AngleInfo *__restrict__ ang, const RayInfo *__restrict__ rays,
          int P, int S, int ba_log2, const float *__restrict__ xb,
          const float *__restrict__ sino, float *__restrict__ out,
          unsigned *__restrict__ maxw) {
  __shared__ unsigned s_max[SB];
  if (MODE != kFwdY) {
    if (threadIdx.x < SB) s_max[threadIdx.x] = 0;
    __syncthreads();
  }
  forward_bundle<SB, MODE, kExact, LPR, kWide>(
      g, ang, rays, P, S, ba_log2, xb, sino, out, s_max,
      xcd_chunked(blockIdx.x, gridDim.x) * (kRayBlock / 64) + (threadIdx.x >> 6), blockIdx.y);
  if (MODE != kFwdY) {
    __syncthreads();
    const int s = blockIdx.y * SB + threadIdx.x;
    if (threadIdx.x < SB && s < S) raise_max(maxw + s, s_max[threadIdx.x]);
  }
}

// w[p][c][s] = r[p][s][c], folding max |r| per slice into maxw (zeroed
// beforehand).  A workgroup transposes blocks of 64 columns x up to 32 slices
// through LDS (rows of 64 floats in, of the slices out) and raises the maxima
// once: 5 slices of 725 columns at 401 angles 96 -> 20 us; before, a workgroup
// took one (p, s) and stored every S-th float.
constexpr int kTransS = 32;
__global__ void __launch_bounds__(256)
k_to_pcs(const float *__restrict__ r, int P, int S, int C, float *__restrict__ w,
         unsigned *__restrict__ maxw) {
  __shared__ float t[kTransS][65];
  __shared__ unsigned s_max[kTransS];
  const int s0 = blockIdx.y * kTransS, ns = min(kTransS, S - s0);
  const int nc = (C + 63) / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned m[kTransS / 4] = {};
  for (int64_t i = blockIdx.x; i < (int64_t)P * nc; i += gridDim.x) {
    const int64_t p = i / nc;
    const int c0 = (int)(i % nc) * 64, cn = min(64, C - c0);
    if (lane < cn) {
#pragma unroll
      for (int j = 0; j < kTransS / 4; ++j) {
        const int s = wave + 4 * j;
        if (s < ns) {
          const float v = r[(p * S + s0 + s) * C + c0 + lane];
          t[s][lane] = v;
          m[j] = max(m[j], __float_as_uint(__builtin_fabsf(v)));
        }
      }
    }
    __syncthreads();
    float *dst = w + (p * C + c0) * S + s0;
    for (int e = threadIdx.x; e < cn * ns; e += 256) {
      const int c = e / ns, s = e - c * ns;
      dst[(int64_t)c * S + s] = t[s][c];
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < kTransS / 4; ++j) {
    for (int off = 32; off > 0; off >>= 1)
      m[j] = max(m[j], (unsigned)__shfl_down((int)m[j], off, 64));
    if (lane == 0) s_max[wave + 4 * j] = m[j];
  }
  __syncthreads();
  if (threadIdx.x < ns) raise_max(maxw + s0 + threadIdx.x, s_max[threadIdx.x]);
}

// ------------------------------------------------------- backprojector --

enum BpMode { kBpSino = 0, kBpOnes = 1, kBpCount = 2 };

struct TileArgs {
  GridInfo g;
  const AngleInfo *ang;
  const RayInfo *rays;
  const int *count;   // [P] upper bound of the columns touching any tile
  int P, S;           // S: slices of a row of w
  int n;              // slices from w, maxw and z on
  int count_lds;      // 1: count[] is staged in LDS after the accumulators
  float yi0;          // detector coordinate of column 0
  const float *w;     // [P][C][S] weights (kBpSino)
  const unsigned *maxw;  // [S] bits of max |w| per slice (kBpSino)
  float maxlen;       // longest segment of the geometry
  float denmax;       // bound on sum of lengths per pixel (max of A^T 1), kBpSino
  float *z;           // [S][N][N] output (kBpOnes/kBpCount: [N][N])
  int wraps;          // some ray has a segment with ix == N (kRayWraps)
  TileSplit split;    // workgroups of a tile (k_bp_tile_split)
};

// LDS accumulator layout of the tile backprojector: one plane per slice,
// rows padded to TW + 1 64-bit words.  Neighbouring rays of one angle sit
// one pixel apart across their direction, so at a given step the lanes of a
// wavefront hit pixels offset by (0, +-1), (+-1, 0) or (+-1, +-1); the odd
// pitch spreads those over the banks.
// Smallest integer whose square is >= v (v >= 0).
constexpr int isqrt_ceil(int v) {
  int q = 0;
  while (q * q < v) ++q;
  return q;
}

template <int TW, int TH>
struct TilePitch {
  static constexpr int kPitch = TW + 1;
  static constexpr int kPlane = TH * kPitch;
};

// Fixed-point accumulation.  LDS float atomics (ds_add_f32) run at a small
// fraction of the rate of LDS integer atomics on gfx950, so each term len*w
// is scaled by 2^e, converted to an integer and added with an integer LDS
// atomic.  Integer addition is associative, so the result does not depend
// on the order in which lanes and waves arrive: the backprojection is
// bit-reproducible.
//   weights (kBpSino): 32-bit words, e per slice such that
//     2^e * max|w| * denmax < 2^30, denmax >= the largest sum of segment
//     lengths in one pixel (max of A^T 1); every pixel's sum then stays
//     below 2^30 + (number of terms)/2, so it cannot overflow; and
//     2^e * max|w| * maxlen < 2^22, so that every term fits the rounding
//     below.  A term is rounded to nearest even with one fma:
//     fl(len * ws + 1.5 * 2^23) is 1.5 * 2^23 + rne(len * ws) exactly (floats
//     in [2^23, 2^24) are the integers), so its bits minus those of
//     1.5 * 2^23 are the integer term (unbiased; error <= 2^-e/2 per term).
//   column sums (kBpOnes): 64-bit words, e from the longest segment
//     (|term| < 2^30), truncated.
// A slice whose weights are not all finite (y = 0 rays give inf/NaN in the
// reference too) is accumulated in float instead, in the same slot, so that
// inf/NaN propagate as they do in the reference.
__device__ __forceinline__ int fixed_exponent(float maxw, float maxlen, bool &fixed) {
  const float m = maxw * maxlen;
  fixed = __builtin_isfinite(m);
  if (!fixed) return 0;
  if (m == 0.f) return 0;
  return 29 - ilogbf(m);
}

constexpr int kNotFixed = INT_MIN;  // exponent of a slice summed in float

// Scale exponent of a weights slice (kBpSino): both bounds above.
__device__ __forceinline__ int weight_exponent(float maxw, float denmax, float maxlen,
                                               bool &fixed) {
  int e = fixed_exponent(maxw, denmax, fixed);
  const float t = maxw * maxlen;
  fixed = fixed && __builtin_isfinite(t);
  if (fixed && t != 0.f) e = min(e, 21 - ilogbf(t));
  return fixed ? e : 0;
}

constexpr float kRoundMagic = 12582912.0f;        // 1.5 * 2^23
constexpr unsigned kRoundMagicBits = 0x4B400000u;  // its bits

// The rounding constant of a slice with scale exponent e, 1.5 * 2^(23 - e):
// fl(len * w + it) is it + 2^-e rne(len * w * 2^e) exactly, so its bits minus
// the constant's are the integer term, without scaling the weights first.
// Its exponent must be a float's (e in [-100, 140]).
__device__ __forceinline__ bool has_magic(int e) { return e >= -100 && e <= 140; }
__device__ __forceinline__ float slice_magic(int e) { return ldexpf(1.5f, 23 - e); }

// Bits of `magic` + rne(len * w) in the last place of a slice's magic.
__device__ __forceinline__ unsigned fixed_bits(float len, float w, float magic) {
  return __float_as_uint(__builtin_fmaf(len, w, magic));
}

// rne(len * ws) as an integer, for |len * ws| < 2^22.
__device__ __forceinline__ int fixed_term(float len, float ws) {
  return (int)(fixed_bits(len, ws, kRoundMagic) - kRoundMagicBits);
}

// Accumulator word of a mode: the weights backprojector sums 32-bit fixed
// point (or float bits for a non-finite slice); column sums and counts use
// 64-bit words.
template <int MODE>
using BpWord = typename std::conditional<MODE == kBpSino, unsigned, unsigned long long>::type;

// Packed weights accumulators (SB >= 2): slices 2k and 2k+1 share a 64-bit
// word, planes [SB/2][TH][TW + 1] of 64-bit words, the even slice in the
// low half, then one plane [TH][TW + 1] of 32-bit per-pixel term counts.
// When every slice of the batch is fixed point, one ds_add_u64 adds both
// terms as the raw fma results: with a, b the rounded terms and M, L the bits
// of the two slices' magics, the 64-bit value 2^32 (L + b) + (M + a) is exact
// (both halves are positive and below 2^31), so after n terms the word holds
// 2^32 (n L + sum b) + n M + sum a (mod 2^64).  Subtracting n (2^32 L + M)
// leaves 2^32 sum(b) + sum(a): its low half is sum(a) (|sum(a)| < 2^31) and
// the rest / 2^32 is sum(b).  A term then costs one fma per slice and the
// two slices one ds_add_u64; the count costs one ds_add_u32 per segment.
// Otherwise each half is its own 32-bit slot (integer or float atomics).
template <int MODE, int SB>
struct BpPacked {
  static constexpr bool value = MODE == kBpSino && SB >= 2 && SB % 2 == 0;
};

// Main loop of the tile backprojector: lanes take consecutive (angle,
// column) pairs of the flattened per-angle column ranges and add their
// segments near the tile into the LDS accumulators.  ALLFX: every slice of
// the batch uses the fixed-point path (the common case; no per-slice
// branch in the inner loop).
//
// The reference's pixel index truncates midpoint + N/2 (trace_utils.cc:
// 177-185), so a segment whose midpoint rounds onto the right image edge
// gets ix == N, i.e. pixel 0 of the next row.  That happens to every
// segment of a near-vertical ray lying within float rounding of the edge
// line x = N/2 (rays on grid lines: an odd C - N, or a half-pixel shift of
// the centre), and such a ray need not pass through the tile that holds
// its target pixels.  pass 0 adds the segments whose midpoint is in the
// tile; pass 1 (EDGE, tiles at column 0 of a geometry with such rays only)
// walks the flagged rays through the strip just left of the right edge,
// rows ty0-1 .. ty1-1, and adds only their wrapped segments.  Each segment
// is added by exactly one pass.
template <int TW, int TH, int SB, int MODE, bool kExact, bool ALLFX, bool EDGE, int BLK>
__device__ __forceinline__ void bp_tile_loop(const TileArgs &a, BpWord<MODE> *acc,
                                             const int *count, int tx0, int tx1, int ty0,
                                             int ty1, int b, const int *ex,
                                             const float (&magic)[SB]) {
  static_assert(SB <= kWeightPad, "a slice batch of weights past the last row must be allocated");
  constexpr int PITCH = TilePitch<TW, TH>::kPitch;
  constexpr int PLANE = TilePitch<TW, TH>::kPlane;
  const int N = a.g.N;
  const int C = a.g.C;
  // region whose rays are walked, and its window in grid lines
  const int wx0 = EDGE ? N - 1 : tx0, wx1 = EDGE ? N : tx1;
  const int wy0 = EDGE ? ty0 - 1 : ty0, wy1 = ty1;
  const float x0 = grid_line(N, wx0), x1 = grid_line(N, wx1);
  const float y0 = grid_line(N, wy0), y1 = grid_line(N, wy1);
  // the strip's column range is at most one wider than a tile's
  constexpr int extra = EDGE ? 1 : 0;
  const bool full = (b + 1) * SB <= a.n;  // no slot past the stack's last slice
  // Lane t takes flat slots t, t + BLK, ... of the tile's (angle,
  // column) pairs.  One slice (kRank): slot f is rank r = f / P of angle
  // p = f % P, rank r being the r-th of the angle's column slots counted
  // from the middle of its range outward, so the lanes of a wavefront take
  // one rank at consecutive angles: rays at the same position relative to
  // the tile, whose two-axis windows have similar lengths.  Several slices:
  // slot f is column slot k of angle p in angle-major order, so the lanes
  // hold neighbouring parallel rays.  Rays of neighbouring angles at the
  // same rank walk nearly the same pixels, and their LDS atomics contend
  // for one address; that costs little with one atomic per segment, and too
  // much with one per slice pair (measured: 15.4 vs 19.8 ms for one
  // 2048^2 slice at 32x32 tiles; 532 vs 109 ms for 64 slices).  One wavefront
  // takes kRankG adjacent ranks, which halves and quarters the lanes that
  // meet at one address.
  constexpr bool kRank = (SB == 1);
  constexpr int kRankG = 4;
  constexpr int kRanks = isqrt_ceil(TW * TW + TH * TH) + 4 + extra;  // >= count[p] + extra
  // Slot iteration: (r, p, k) -> the lane's next (angle, column slot).
  auto advance = [&](int &r, int &p, int &k) {
    if (kRank) {
      p += BLK / kRankG;
      while (p >= a.P) { p -= a.P; r += kRankG; }
    } else {
      k += BLK;
      while (p < a.P && k >= count[p] + extra) { k -= count[p] + extra; ++p; }
    }
  };
  auto live = [&](int r, int p) { return kRank ? r < kRanks : p < a.P; };
  // One (angle, column) pair, fetched a pair ahead of its walk: the ray
  // table entry and the weights mostly miss L2, so their loads for the next
  // pair are in flight while the current pair is walked.
  struct Pair {
    bool ok;
    int quadrant;
    RayInfo ray;
    float w[SB];
  };
  // A pair's slot resolved to (angle, column slot), and whether it exists
  // so far (the column range is checked when the pair is fetched).
  struct Slot {
    int p, k;
    bool ok;
  };
  auto resolve = [&](int r, int p, int k) {
    const bool lv = live(r, p);
    Slot o{lv ? p : 0, k, lv};
    if (kRank) {
      const int cnt = count[o.p] + extra;
      o.ok = o.ok && r < cnt;
      o.k = ((cnt - 1) >> 1) + ((r & 1) ? (r + 1) >> 1 : -(r >> 1));
    }
    return o;
  };
  // Every lane issues the same loads on every path (row 0 when it has no
  // pair; a whole slice batch of weights, which the kWeightPad floats after
  // the weights keep in bounds for the last row): with one path, the
  // compiler's wait for the current pair's data covers that pair only, and
  // not the next pair's loads issued after it.  The angle record comes in
  // loaded a pair earlier still, so no wait at all sits between a pair's
  // resolution and its loads.
  auto fetch = [&](const Slot &sl, const AngleInfo &ang, Pair &q) {
    const int pp = sl.p, k = sl.k;
    bool ok = sl.ok;
    int cmin, cmax;
    tile_columns(ang, x0, x1, y0, y1, a.yi0, cmin, cmax);
    const int c = cmin + k;
    ok = ok && c >= 0 && c < C && c <= cmax;
    q.ok = ok;
    q.quadrant = ang.quadrant;
    const int64_t t = ok ? (int64_t)pp * C + c : 0;
    q.ray = a.rays[t];
    if (MODE == kBpSino) {
      const float *wr = a.w + t * a.S + b * SB;
      if constexpr (SB % 4 == 0) {
#pragma unroll
        for (int i = 0; i < SB; i += 4) {
          float4 v;
          __builtin_memcpy(&v, wr + i, sizeof v);  // rows are 4-byte aligned
          q.w[i] = v.x, q.w[i + 1] = v.y, q.w[i + 2] = v.z, q.w[i + 3] = v.w;
        }
      } else {
#pragma unroll
        for (int i = 0; i < SB; ++i) q.w[i] = wr[i];
      }
    }
  };
  int r = 0, p = 0, k = threadIdx.x;
  if (kRank) {
    const int g = threadIdx.x / kRankG;
    r = g / a.P * kRankG + threadIdx.x % kRankG;
    p = g % a.P;
  } else {
    while (p < a.P && k >= count[p] + extra) { k -= count[p] + extra; ++p; }
  }
  Pair cur;
  {
    const Slot s0 = resolve(r, p, k);
    fetch(s0, a.ang[s0.p], cur);
  }
  int rn = r, pn = p, kn = k;
  advance(rn, pn, kn);
  Slot sn = resolve(rn, pn, kn);
  AngleInfo angn = a.ang[sn.p];
  while (live(r, p)) {
    // the pair after next: slot and angle record
    int rnn = rn, pnn = pn, knn = kn;
    advance(rnn, pnn, knn);
    const Slot snn = resolve(rnn, pnn, knn);
    const AngleInfo angnn = a.ang[snn.p];
    Pair nxt;
    fetch(sn, angn, nxt);
    if (cur.ok) {
      // ALLFX takes the weights as they are and rounds by the slices' magics;
      // otherwise they are pre-scaled by 2^e (exact: a power-of-two scaling
      // commutes with rounding, so fl(len * ws) = fl(len * w) * 2^e)
      float wv[SB];
      bool any = true;
      if (MODE == kBpSino) {
        unsigned nz = 0;
#pragma unroll
        for (int q = 0; q < SB; ++q) {
          // slots past the stack's last slice (read from the next row) add 0
          const float wq = full || b * SB + q < a.n ? cur.w[q] : 0.f;
          nz |= __float_as_uint(wq);
          wv[q] = (!ALLFX && ex[q] != kNotFixed) ? ldexpf(wq, ex[q]) : wq;
        }
        any = (nz << 1) != 0;  // some weight is not +-0
      } else if (MODE == kBpOnes) {
        wv[0] = ldexpf(1.0f, ex[0]);
      }
      if (any && (!EDGE || (cur.ray.alo & kRayWraps))) {
        traverse_window<kExact, kRank>(a.g, cur.ray, cur.quadrant, wx0, wx1, wy0, wy1,
                                [&](int ix, int iy, float l, float) {
          // ix == N is pixel 0 of the next row (truncation).  The edge pass
          // takes those segments; the others reject them, as no tile has a
          // pixel column N (a cell past the image in a tile cut by its edge
          // is summed but not written out).
          bool in;
          unsigned lx, ly;
          if constexpr (EDGE) {
            lx = 0;
            ly = (unsigned)(iy + 1 - ty0);
            in = ix == N && ly < (unsigned)(ty1 - ty0);
          } else {
            lx = (unsigned)(ix - tx0);
            ly = (unsigned)(iy - ty0);
            in = lx < (unsigned)TW && ly < (unsigned)TH;
          }
          if (in) {
            const unsigned cell = __umul24(ly, PITCH) + lx;
            BpWord<MODE> *dst = acc + cell;
            if (MODE == kBpCount) {
              atomicAdd(dst, (BpWord<MODE>)1);
            } else if (MODE == kBpOnes) {
              // |t| < 2^30: truncating conversion, error < 2^-e
              atomicAdd(dst, (BpWord<MODE>)(long long)(int)(l * wv[0]));
            } else if (BpPacked<MODE, SB>::value) {
              // 32-bit index of the pixel's 64-bit word in pair plane 0
              unsigned *d2 = reinterpret_cast<unsigned *>(acc) + 2 * cell;
#pragma unroll
              for (int k2 = 0; k2 < SB / 2; ++k2) {
                unsigned *dk = d2 + 2 * k2 * PLANE;
                if (ALLFX) {
                  const unsigned long long v =
                      ((unsigned long long)fixed_bits(l, wv[2 * k2 + 1], magic[2 * k2 + 1])
                       << 32) |
                      fixed_bits(l, wv[2 * k2], magic[2 * k2]);
                  atomicAdd(reinterpret_cast<unsigned long long *>(dk), v);
                } else {
#pragma unroll
                  for (int h = 0; h < 2; ++h) {
                    const int q = 2 * k2 + h;
                    if (ex[q] != kNotFixed)
                      atomicAdd(dk + h, (unsigned)fixed_term(l, wv[q]));
                    else
                      atomicAdd(reinterpret_cast<float *>(dk + h), l * wv[q]);
                  }
                }
              }
              // terms per pixel, for the magic offsets of the ALLFX words
              if (ALLFX)
                atomicAdd(reinterpret_cast<unsigned *>(acc) + SB * PLANE + cell, 1u);
            } else {
#pragma unroll
              for (int q = 0; q < SB; ++q) {
                if (ALLFX) {
                  atomicAdd(dst + q * PLANE, (BpWord<MODE>)(fixed_bits(l, wv[q], magic[q]) -
                                                            __float_as_uint(magic[q])));
                } else if (ex[q] != kNotFixed) {
                  atomicAdd(dst + q * PLANE, (BpWord<MODE>)fixed_term(l, wv[q]));
                } else {
                  atomicAdd(reinterpret_cast<float *>(dst + q * PLANE), l * wv[q]);
                }
              }
            }
          }
        });
      }
    }
    r = rn;
    p = pn;
    k = kn;
    cur = nxt;
    rn = rnn;
    pn = pnn;
    kn = knn;
    sn = snn;
    angn = angnn;
  }
}

// LDS words (BpWord<MODE>) of a tile's accumulators: the slice planes, and
// for packed weights the per-pixel term counts.
template <int TW, int TH, int SB, int MODE>
constexpr int bp_acc_words() {
  return (SB + (BpPacked<MODE, SB>::value ? 1 : 0)) * TilePitch<TW, TH>::kPlane;
}

// Workgroup (tile, slice batch): LDS accumulators acc[SB][TH][TW + 1] for
// all angles, then one coalesced write-out.  `acc` is the workgroup's
// dynamic LDS (bp_acc_words() words of BpWord<MODE>, then int count[P]
// when a.count_lds); the body starts and ends with a workgroup barrier, so a
// persistent workgroup may run it for one tile after another.
//
// kSplit: this workgroup has taken a share of the angles (a is narrowed to
// it), `part` is its place among the a.split.n partial accumulators of the
// tile, and the workgroup that finishes last adds the others' and writes out.
// The words are integers, so their sum does not depend on the split.  A batch
// with a non-finite slice is summed in float; `whole` then holds all angles
// for the first workgroup.
template <int TW, int TH, int SB, int MODE, bool kExact, int BLK, bool kSplit = false>
__device__ __forceinline__ void bp_tile_body(TileArgs a, int tile, int b,
                                             unsigned long long *lds, int part = 0,
                                             const TileArgs *whole = nullptr) {
  BpWord<MODE> *acc = reinterpret_cast<BpWord<MODE> *>(lds);
  constexpr int PITCH = TilePitch<TW, TH>::kPitch;
  constexpr int PLANE = TilePitch<TW, TH>::kPlane;
  constexpr int WORDS = bp_acc_words<TW, TH, SB, MODE>();
  int *lcount = reinterpret_cast<int *>(acc + WORDS);
  const int *count = !kSplit && a.count_lds ? lcount : a.count;
  const int N = a.g.N;
  const int tiles_x = (N + TW - 1) / TW;
  const int tx = tile % tiles_x, ty = tile / tiles_x;
  const int tx0 = tx * TW, ty0 = ty * TH;
  const int tx1 = min(tx0 + TW, N), ty1 = min(ty0 + TH, N);
  __syncthreads();  // the previous tile's write-out has read acc and s_ex
  for (int i = threadIdx.x; i < WORDS; i += BLK) acc[i] = 0;
  if (!kSplit && a.count_lds)
    for (int i = threadIdx.x; i < a.P; i += BLK) lcount[i] = a.count[i];
  // Per-slice scale exponents (kNotFixed: a float slice) in LDS, where the
  // write-out and the mixed form read them; the all-fixed loop takes the
  // slices' magics, uniform, straight into its fused multiply-adds (kept per
  // slice with a flag each, they spilled 400 scalar registers at 32 slices).
  __shared__ int s_ex[SB];
  bool fixed = true;
  if (threadIdx.x < SB) {
    const int s = b * SB + (int)threadIdx.x;
    int e;
    if (MODE == kBpSino)
      e = weight_exponent((s < a.n) ? __uint_as_float(a.maxw[s]) : 0.f, a.denmax, a.maxlen,
                          fixed);
    else
      e = fixed_exponent(1.0f, a.maxlen, fixed);
    s_ex[threadIdx.x] = fixed ? e : kNotFixed;
    fixed = fixed && (MODE != kBpSino || has_magic(e));
  }
  const bool all_fixed = __syncthreads_and(fixed);
  if constexpr (kSplit) {
    if (!all_fixed) {
      if (part != 0) return;
      a = *whole;
    }
    count = a.count;
  }
  float magic[SB];
#pragma unroll
  for (int q = 0; q < SB; ++q) {
    magic[q] = slice_magic(all_fixed ? s_ex[q] : 0);
    // scalar registers hold up to 16 of them beside the rest
    if constexpr (SB <= 16)
      magic[q] = __uint_as_float((unsigned)__builtin_amdgcn_readfirstlane(
          (int)__float_as_uint(magic[q])));
  }
  if (MODE == kBpCount || all_fixed) {
    bp_tile_loop<TW, TH, SB, MODE, kExact, true, false, BLK>(a, acc, count, tx0, tx1, ty0, ty1, b,
                                                        s_ex, magic);
    if (tx0 == 0 && a.wraps)
      bp_tile_loop<TW, TH, SB, MODE, kExact, true, true, BLK>(a, acc, count, tx0, tx1, ty0, ty1, b,
                                                         s_ex, magic);
  } else {
    bp_tile_loop<TW, TH, SB, MODE, kExact, false, false, BLK>(a, acc, count, tx0, tx1, ty0, ty1, b,
                                                         s_ex, magic);
    if (tx0 == 0 && a.wraps)
      bp_tile_loop<TW, TH, SB, MODE, kExact, false, true, BLK>(a, acc, count, tx0, tx1, ty0, ty1, b,
                                                          s_ex, magic);
  }
  __syncthreads();
  if constexpr (kSplit) {
    if (all_fixed) {
      static_assert(sizeof(BpWord<MODE>) == 4, "32-bit words");
      const int64_t item = (int64_t)b * gridDim.x + tile;
      unsigned *parts = a.split.part + item * a.split.n * WORDS;
      // Every wavefront's stores are complete at the barrier; the release on the
      // ticket then publishes the workgroup's words to the GPU, and the acquire
      // of the workgroup that takes the last ticket sees those of all before it
      // (each ticket's release goes on in the read-modify-writes that follow it).
      // The words go past the XCD's L2 besides (agent scope), which leaves the
      // release little to write back.
      for (int i = threadIdx.x; i < WORDS; i += BLK)
        __hip_atomic_store(parts + (int64_t)part * WORDS + i, (unsigned)acc[i], __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      wait_vector_loads();  // loads and stores share the counter
      __shared__ int s_last;
      __syncthreads();
      if (threadIdx.x == 0) {
        unsigned *ticket = a.split.ticket + item;
        s_last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT) ==
                 (unsigned)(a.split.n - 1);
        if (s_last) {
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
          atomicExch(ticket, 0u);  // for the next launch
        }
      }
      __syncthreads();
      if (!s_last) return;
      auto get = [](const unsigned *p) {
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      };
      constexpr int PAIRS = BpPacked<MODE, SB>::value ? SB / 2 * PLANE : 0;  // 64-bit words
      unsigned long long *acc64 = reinterpret_cast<unsigned long long *>(acc);
      for (int k = 0; k < a.split.n; ++k) {
        if (k == part) continue;
        const unsigned *src = parts + (int64_t)k * WORDS;
        for (int i = threadIdx.x; i < PAIRS; i += BLK)
          acc64[i] += ((unsigned long long)get(src + 2 * i + 1) << 32) | get(src + 2 * i);
        for (int i = 2 * PAIRS + threadIdx.x; i < WORDS; i += BLK) acc[i] += get(src + i);
      }
      __syncthreads();
    }
  }
  // coalesced write-out: plane by plane, row-contiguous
  const int w_ = tx1 - tx0, h_ = ty1 - ty0;
  if (BpPacked<MODE, SB>::value) {
    const unsigned long long *acc64 = reinterpret_cast<const unsigned long long *>(acc);
    const unsigned *nterms = reinterpret_cast<const unsigned *>(acc) + SB * PLANE;
#pragma unroll
    for (int k2 = 0; k2 < SB / 2; ++k2) {
      for (int i = threadIdx.x; i < w_ * h_; i += BLK) {
        const int ly = i / w_, lx = i - ly * w_;
        unsigned long long v = acc64[k2 * PLANE + ly * PITCH + lx];
        // remove the magic offsets, n times both slices' bits, mod 2^64
        if (all_fixed)
          v -= (unsigned long long)nterms[ly * PITCH + lx] *
               (((unsigned long long)__float_as_uint(magic[2 * k2 + 1]) << 32) |
                __float_as_uint(magic[2 * k2]));
        const int lo = (int)(unsigned)v;
        const int hi = (int)(((long long)v - (long long)lo) >> 32);
        const int64_t o = (int64_t)(ty0 + ly) * N + tx0 + lx;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int q = 2 * k2 + h;
          const int s = b * SB + q;
          if (s >= a.n) break;
          const unsigned half = h ? (unsigned)(v >> 32) : (unsigned)v;
          float out;
          if (s_ex[q] == kNotFixed)
            out = __uint_as_float(half);
          else
            out = (float)ldexp((double)(all_fixed ? (h ? hi : lo) : (int)half), -s_ex[q]);
          a.z[(int64_t)s * N * N + o] = out;
        }
      }
    }
    return;
  }
#pragma unroll
  for (int q = 0; q < SB; ++q) {
    const int s = b * SB + q;
    if (MODE == kBpSino && s >= a.n) break;
    float *zs = a.z + (int64_t)s * N * N;
    for (int i = threadIdx.x; i < w_ * h_; i += BLK) {
      const int ly = i / w_, lx = i - ly * w_;
      const BpWord<MODE> v = acc[q * PLANE + ly * PITCH + lx];
      float out;
      if (MODE == kBpCount)
        out = (float)v;
      else if (s_ex[q] == kNotFixed)
        out = __uint_as_float((unsigned)v);
      else if (MODE == kBpSino)
        out = (float)ldexp((double)(int)v, -s_ex[q]);
      else
        out = (float)ldexp((double)(long long)v, -s_ex[q]);
      zs[(int64_t)(ty0 + ly) * N + tx0 + lx] = out;
    }
  }
}

template <int TW, int TH, int SB, int MODE, bool kExact, int BLK>
__global__ void __launch_bounds__(BLK)
k_bp_tile(TileArgs a) {
  extern __shared__ unsigned long long acc[];
  bp_tile_body<TW, TH, SB, MODE, kExact, BLK>(a, blockIdx.x, blockIdx.y, acc);
}

// The angles of a tile shared among a.split.n workgroups (blockIdx.z), for
// images with fewer tiles than the GPU has CUs.
template <int TW, int TH, int SB, bool kExact, int BLK>
__global__ void __launch_bounds__(BLK)
k_bp_tile_split(TileArgs all) {
  extern __shared__ unsigned long long acc[];
  TileArgs a = all;
  const int per = (all.P + all.split.n - 1) / all.split.n;
  const int p0 = (int)blockIdx.z * per;
  a.P = min(per, all.P - p0);  // at least one (tile_splits)
  a.ang += p0;
  a.count += p0;
  a.rays += (int64_t)p0 * a.g.C;
  a.w += (int64_t)p0 * a.g.C * a.S;
  bp_tile_body<TW, TH, SB, kBpSino, kExact, BLK, true>(a, blockIdx.x, blockIdx.y, acc,
                                                       (int)blockIdx.z, &all);
}

// Per-slice maximum of |w| over w [P][C][S] (float bits, atomicMax on the
// non-negative bit patterns; NaN sorts above inf).  maxw must be zeroed.
__global__ void __launch_bounds__(kPixBlock)
k_absmax_slices(const float *__restrict__ w, int P, int S, int C, unsigned *__restrict__ maxw) {
  const int s = blockIdx.y;
  const int64_t n = (int64_t)P * C;
  unsigned m = 0;
  for (int64_t i = (int64_t)blockIdx.x * kPixBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kPixBlock)
    m = max(m, __float_as_uint(__builtin_fabsf(w[i * S + s])));
  __shared__ unsigned s_max[kPixBlock / 64];
  for (int off = 32; off > 0; off >>= 1) m = max(m, (unsigned)__shfl_down((int)m, off, 64));
  if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < kPixBlock / 64; ++k) m = max(m, s_max[k]);
    raise_max(maxw + s, m);
  }
}

// ------------------------------------------------------- pack / update --

// xb[t/SB][j][t%SB] = src[(t + off)][j] for t < S_src_used, ghost value
// outside: slots whose source slice index is < 0 or >= nsrc get `fill`.
template <int SB>
__global__ void __launch_bounds__(kPixBlock)
k_pack(const float *__restrict__ src, int nsrc, int off, float fill, int64_t NN, int nslots,
       float *__restrict__ xb) {
  const int64_t j = (int64_t)blockIdx.x * kPixBlock + threadIdx.x;
  const int b = blockIdx.y;
  if (j >= NN) return;
  float v[SB];
#pragma unroll
  for (int q = 0; q < SB; ++q) {
    const int t = b * SB + q;
    const int s = t + off;
    v[q] = (t < nslots && s >= 0 && s < nsrc) ? src[(int64_t)s * NN + j] : fill;
  }
  float *dst = xb + ((int64_t)b * NN + j) * SB;
  store_slices<SB>(dst, v);
}

// The updates run between the backprojector, which reads the slices' largest
// weights, and the next projection, which gathers them anew: their first
// workgroup clears them (a launch for it took 4 us an iteration).
__device__ __forceinline__ void clear_max(unsigned *maxw, int S) {
  if ((blockIdx.x | blockIdx.y | blockIdx.z) == 0)
    for (int s = threadIdx.x; s < S; s += kPixBlock) maxw[s] = 0;
}

// SIRT (sirt.cc:21-33) / MLEM (mlem.cc:21-34) update of VB slices of a batch
// at pixel j, also refreshing the batched copy (with one slice to a batch x
// is that copy).
template <int SB, int VB, bool kSIRT>
__global__ void __launch_bounds__(kPixBlock)
k_update_em(float *__restrict__ x, const float *__restrict__ z, const float *__restrict__ den,
            int S, int64_t NN, float *__restrict__ xb, unsigned *__restrict__ maxw) {
  const int64_t j = (int64_t)blockIdx.x * kPixBlock + threadIdx.x;
  const int s0 = blockIdx.y * VB;
  clear_max(maxw, S);
  if (j >= NN) return;
  const float d = den[j];
  float v[VB];
#pragma unroll
  for (int q = 0; q < VB; ++q) {
    const int s = s0 + q;
    v[q] = 0.f;
    if (s < S) {
      const int64_t o = (int64_t)s * NN + j;
      float xv = x[o];
      if (kSIRT) xv += z[o] / d;
      else xv *= z[o] / d;
      x[o] = xv;
      v[q] = xv;
    }
  }
  if (SB > 1) store_slices<VB>(xb + ((int64_t)(s0 / SB) * NN + j) * SB + s0 % SB, v);
}

__global__ void k_fill(float *__restrict__ p, int64_t n, float v) {
  const int64_t i = (int64_t)blockIdx.x * kPixBlock + threadIdx.x;
  if (i < n) p[i] = v;
}

// Pixel classes and neighbour orders of the regularisation stencils:
// 0 inner, 1 top row, 2 bottom row, 3 left column, 4 right column,
// 5..8 corners top-left, top-right, bottom-left, bottom-right.  The in-plane
// neighbour order per class is the reference's q order (pml.cc:45-53,
// 69-74, 87-92, 105-110, 123-128, 141-144, 156-159, 171-174, 187-190; the
// same orders appear in apmlr.cc).
__constant__ int8_t c_nb[9][8][2] = {
    {{1, 0}, {-1, 0}, {0, 1}, {0, -1}, {1, 1}, {-1, 1}, {1, -1}, {-1, -1}},
    {{1, 0}, {-1, 0}, {0, 1}, {1, 1}, {-1, 1}},
    {{1, 0}, {-1, 0}, {0, -1}, {1, -1}, {-1, -1}},
    {{1, 0}, {0, 1}, {0, -1}, {1, 1}, {1, -1}},
    {{-1, 0}, {0, 1}, {0, -1}, {-1, 1}, {-1, -1}},
    {{1, 0}, {0, 1}, {1, 1}},
    {{-1, 0}, {0, 1}, {-1, 1}},
    {{1, 0}, {0, -1}, {1, -1}},
    {{-1, 0}, {0, -1}, {-1, -1}},
};
__constant__ int c_nbn[9] = {8, 5, 5, 5, 5, 3, 3, 3, 3};

// PML weights, pml.h:22-29
__constant__ float c_pml_w[3][8] = {
    {0.1464466094f, 0.1464466094f, 0.1464466094f, 0.1464466094f,
     0.10355339059f, 0.10355339059f, 0.10355339059f, 0.10355339059f},
    {0.226540919667f, 0.226540919667f, 0.226540919667f, 0.1601886205f,
     0.1601886205f},
    {0.36939806251f, 0.36939806251f, 0.26120387496f}};

__device__ __forceinline__ int pixel_class(int m, int n, int N) {
  const bool top = (n == 0), bot = (n == N - 1), left = (m == 0),
             right = (m == N - 1);
  if (!(top | bot | left | right)) return 0;
  if (top && left) return 5;
  if (top && right) return 6;
  if (bot && left) return 7;
  if (bot && right) return 8;
  if (top) return 1;
  if (bot) return 2;
  if (left) return 3;
  return 4;
}

// In-plane neighbour offsets and PML weights of an inner pixel, in the
// reference's q order (pml.cc:45-53, the first row of c_nb and c_pml_w),
// as compile-time constants: inner pixels (all but the border) skip the
// per-class tables.
constexpr int kInnerDx[8] = {1, -1, 0, 0, 1, -1, 1, -1};
constexpr int kInnerDy[8] = {0, 0, 1, -1, 1, 1, -1, -1};
constexpr float kPmlAxial = 0.1464466094f;
constexpr float kPmlDiag = 0.10355339059f;

// PML stencil and update of the VB slices from s0 on at one pixel.
template <int VB, bool kInner>
__device__ __forceinline__ void pml_pixel(const float *__restrict__ x, float *__restrict__ xn,
                                          const float *__restrict__ z, int S, int N,
                                          int64_t NN, int64_t pix, int cls, float d,
                                          float beta, int num_direct, int s0, float (&v)[VB]) {
  const float *w = c_pml_w[cls == 0 ? 0 : (cls <= 4 ? 1 : 2)];
  const int cnt = c_nbn[cls];
#pragma unroll
  for (int q = 0; q < VB; ++q) {
    const int s = s0 + q;
    v[q] = 0.f;
    if (s < S) {
      const int64_t j = (int64_t)s * NN + pix;
      const float x0 = x[j];
      float f = 0.f, gg = 0.f;
      if (kInner) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float xq = x[j + kInnerDx[k] + (int64_t)kInnerDy[k] * N];
          const float wk = k < 4 ? kPmlAxial : kPmlDiag;
          f += 2.0f * beta * wk;
          gg -= 2.0f * beta * wk * (x0 + xq);
        }
      } else {
        for (int k = 0; k < cnt; ++k) {
          const float xq = x[j + c_nb[cls][k][0] + (int64_t)c_nb[cls][k][1] * N];
          f += 2.0f * beta * w[k];
          gg -= 2.0f * beta * w[k] * (x0 + xq);
        }
      }
      const float G = gg + d;
      const float F = f;
      const float nm = num_direct ? z[j] : -(x0 * z[j]);
      const float xv = (-G + __builtin_sqrtf(G * G - 8.0f * nm * F)) / (4.0f * F);
      xn[j] = xv;
      v[q] = xv;
    }
  }
}

// Fused PML stencil (pml.cc:25-201, F and G from zero) and closed-form
// update (pml.cc:3-23):  x' = (-G + sqrt(G^2 - 8 num F)) / (4F).  With
// num_direct, z holds num as the reference sums it (ordered.hip); otherwise
// z = A^T w and num = -x * z (the x factor of pml.cc:243 taken out of the
// sum).
// A thread owns a pixel of VB of the SB slices of a slot batch and also
// writes their part of the slice-batched copy xb of the new image for the next
// ray pass (slot t = slice t; padding slots hold 0).
template <int SB, int VB>
__global__ void __launch_bounds__(kPixBlock)
k_update_pml(const float *__restrict__ x, float *__restrict__ xn,
             const float *__restrict__ z, const float *__restrict__ den,
             int S, int N, float beta, int num_direct, float *__restrict__ xb,
             unsigned *__restrict__ maxw) {
  const int pix = blockIdx.x * kPixBlock + threadIdx.x;
  const int s0 = blockIdx.y * VB;
  clear_max(maxw, S);
  if (pix >= N * N) return;
  const int64_t NN = (int64_t)N * N;
  const int n = pix / N, m = pix - n * N;
  const int cls = pixel_class(m, n, N);
  const float d = den[pix];
  float v[VB];
  if (cls == 0)
    pml_pixel<VB, true>(x, xn, z, S, N, NN, pix, cls, d, beta, num_direct, s0, v);
  else
    pml_pixel<VB, false>(x, xn, z, S, N, NN, pix, cls, d, beta, num_direct, s0, v);
  store_slices<VB>(xb + ((int64_t)(s0 / SB) * NN + pix) * SB + s0 % SB, v);
}

struct ApmlrArgs {
  StencilWeights w;
  RegParams p;
  int compat;
  int nslots;      // slots of the batched copy
  int num_direct;  // z holds num (ordered.hip), not A^T w
};

// APMLR stencil and update of the VB slots from t0 on at one pixel (see
// k_update_apmlr).
template <int VB, bool kInner>
__device__ __forceinline__ void apmlr_pixel(const float *__restrict__ xp,
                                            float *__restrict__ xnp,
                                            const float *__restrict__ z, int S, int N,
                                            int64_t NN, int64_t pix, int cls, float d,
                                            const ApmlrArgs &a, int t0, float (&v)[VB]) {
  const int cnt = kInner ? 8 : c_nbn[cls];
  const int off = a.compat ? 0 : 1;
  const float tb = 2.0f * a.p.beta;
  const float tb1 = 2.0f * a.p.beta1;
#pragma unroll
  for (int q = 0; q < VB; ++q) {
    const int pi = t0 + q + off;  // padded slice of slot t0 + q
    float val = 0.f;
    if (pi >= 1 && pi <= S) {
      const int s = pi - 1;
      const int64_t jp = (int64_t)pi * NN + pix;
      const int64_t j = (int64_t)s * NN + pix;
      const bool top = (s == 0), bottom = (s == S - 1 && S - 1 != 0);
      const int zmode = top ? 1 : (bottom ? 2 : 0);
      const int nz = zmode == 0 ? 2 : 1;
      const float *w = a.w.w[zmode][kInner ? 0 : cls];
      const float x0 = xp[jp];
      float f = 0.f, gg = 0.f;
      if (kInner) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float xq = xp[jp + kInnerDx[k] + (int64_t)kInnerDy[k] * N];
          const float mg = x0 + xq;
          const float rg = x0 - xq;
          const float gm = 1.0f / (1.0f + __builtin_fabsf(rg / a.p.delta));
          f += tb * w[k] * gm;
          gg -= tb * w[k] * gm * mg;
        }
      } else {
        for (int k = 0; k < cnt; ++k) {
          const float xq = xp[jp + c_nb[cls][k][0] + (int64_t)c_nb[cls][k][1] * N];
          const float mg = x0 + xq;
          const float rg = x0 - xq;
          const float gm = 1.0f / (1.0f + __builtin_fabsf(rg / a.p.delta));
          f += tb * w[k] * gm;
          gg -= tb * w[k] * gm * mg;
        }
      }
      for (int k = 0; k < nz; ++k) {
        const int64_t dz = (zmode == 2 || k == 1) ? -NN : NN;
        const float xq = xp[jp + dz];
        const float mg = x0 + xq;
        const float rg = x0 - xq;
        const float gm = 1.0f / (1.0f + __builtin_fabsf(rg / a.p.delta1));
        f += tb1 * w[cnt + k] * gm;
        gg -= tb1 * w[cnt + k] * gm * mg;
      }
      const float G = gg + d;
      const float F = f;
      const float xpass = a.compat ? xp[jp - NN] : x0;
      const float nm = a.num_direct ? z[j] : -(xpass * z[j]);
      val = (-G + __builtin_sqrtf(G * G - 8.0f * nm * F)) / (4.0f * F);
      xnp[jp] = val;
    } else if (pi == 0 || pi == S + 1) {
      val = xp[(int64_t)pi * NN + pix];
    }
    v[q] = val;
  }
}

// Fused APMLR stencil (apmlr.cc:919-982 with FGInner/FGTop/FGBottom) and
// update (apmlr.cc:3-26) over ghost-padded images [S+2][N][N]; real slice s
// lives at padded index s+1.  The ray pass of slice s used padded slice s
// (compat, apmlr.cc:1082-1084) or s+1, which also supplies num's x factor.
// Thread (pixel, VB slots of a slot batch): slot t of the batched copy holds
// padded slice t + off (off = 0 compat, 1 otherwise); real slices are updated,
// ghosts (padded 0 and S+1, constant) are copied, slots past S+1 hold 0.
// The grid covers every real slice even when its slot lies past nslots.
template <int SB, int VB>
__global__ void __launch_bounds__(kPixBlock)
k_update_apmlr(const float *__restrict__ xp, float *__restrict__ xnp,
               const float *__restrict__ z, const float *__restrict__ den,
               int S, int N, ApmlrArgs a, float *__restrict__ xb,
               unsigned *__restrict__ maxw) {
  const int pix = blockIdx.x * kPixBlock + threadIdx.x;
  const int t0 = blockIdx.y * VB;
  clear_max(maxw, S);
  if (pix >= N * N) return;
  const int64_t NN = (int64_t)N * N;
  const int n = pix / N, m = pix - n * N;
  const int cls = pixel_class(m, n, N);
  const float d = den[pix];
  float v[VB];
  if (cls == 0)
    apmlr_pixel<VB, true>(xp, xnp, z, S, N, NN, pix, cls, d, a, t0, v);
  else
    apmlr_pixel<VB, false>(xp, xnp, z, S, N, NN, pix, cls, d, a, t0, v);
  if (t0 < a.nslots) store_slices<VB>(xb + ((int64_t)(t0 / SB) * NN + pix) * SB + t0 % SB, v);
}

// ------------------------------------------------------------- batched --
//
// Persistent kernels over the work queues of a batch of slices with
// different geometries (BatchQueues).  Each workgroup takes an item, finds
// its slice by binary search in the phase's start table and runs the same
// per-item code as the single-geometry kernels (one slice per geometry).

__device__ __forceinline__ int batch_next_item(unsigned *counter) {
  __shared__ unsigned s_item;
  __syncthreads();  // every lane has read the previous item
  if (threadIdx.x == 0) s_item = atomicAdd(counter, 1u);
  __syncthreads();
  return __builtin_amdgcn_readfirstlane((int)s_item);
}

__device__ __forceinline__ int batch_find(const int *__restrict__ start, int n, int item) {
  int lo = 0, hi = n;  // start[lo] <= item < start[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (start[mid] <= item) lo = mid;
    else hi = mid;
  }
  return lo;
}

__global__ void k_batch_reset(unsigned *__restrict__ counters, unsigned *__restrict__ maxw,
                              int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 3) counters[i] = 0u;
  if (i < n) maxw[i] = 0u;
}

template <bool kExact>
__global__ void __launch_bounds__(kRayBlock)
k_forward_batch(const BatchSliceDev *__restrict__ d, BatchQueues q, int it, int ba_log2) {
  const int *start = q.start[0];
  const int total = start[q.n];
  __shared__ unsigned s_max[1];
  if (threadIdx.x == 0) s_max[0] = 0;  // the next barrier: batch_next_item's
  for (;;) {
    const int item = batch_next_item(q.counters + 0);
    if (item >= total) break;
    const int k = batch_find(start, q.n, item);
    const BatchSliceDev &sd = d[__builtin_amdgcn_readfirstlane(q.order[0][k])];
    if (it >= sd.iters) continue;
    const int64_t bundle = (int64_t)(item - start[k]) * (kRayBlock / 64) + (threadIdx.x >> 6);
    auto run = [&](auto mode, auto wide) {
      forward_bundle<1, decltype(mode)::value, kExact, 1, decltype(wide)::value>(
          sd.g, sd.ang, sd.rays, sd.P, 1, ba_log2, sd.x, sd.sino, sd.w, s_max, bundle, 0);
    };
    using std::integral_constant;
    if (wide_image(sd.g.N, 1)) {
      if (sd.alg == 0) run(integral_constant<int, kFwdSIRT>(), std::true_type());
      else run(integral_constant<int, kFwdEM>(), std::true_type());
    } else if (sd.alg == 0) {
      run(integral_constant<int, kFwdSIRT>(), std::false_type());
    } else {
      run(integral_constant<int, kFwdEM>(), std::false_type());
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      raise_max(sd.maxw, s_max[0]);
      s_max[0] = 0;
    }
  }
}

template <int TW, int TH, bool kExact>
__global__ void __launch_bounds__(kTileBlock)
k_bp_batch(const BatchSliceDev *__restrict__ d, BatchQueues q, int it) {
  extern __shared__ unsigned long long acc[];  // [TH][TW + 1], then int count[P]
  const int *start = q.start[1];
  const int total = start[q.n];
  for (;;) {
    const int item = batch_next_item(q.counters + 1);
    if (item >= total) break;
    const int k = batch_find(start, q.n, item);
    const BatchSliceDev &sd = d[__builtin_amdgcn_readfirstlane(q.order[1][k])];
    if (it >= sd.iters) continue;
    TileArgs a;
    a.g = sd.g;
    a.ang = sd.ang;
    a.rays = sd.rays;
    a.count = sd.count;
    a.P = sd.P;
    a.S = a.n = 1;
    a.count_lds = 1;
    a.yi0 = sd.yi0;
    a.w = sd.w;
    a.maxw = sd.maxw;
    a.maxlen = sd.maxlen;
    a.denmax = sd.denmax;
    a.z = sd.z;
    a.wraps = sd.wraps;
    bp_tile_body<TW, TH, 1, kBpSino, kExact, kTileBlock>(a, item - start[k], 0, acc);
  }
}

// SIRT (sirt.cc:21-33) / MLEM (mlem.cc:21-34) update, kBatchUpdateBlocks
// blocks of kPixBlock pixels per item (one item per block made the shared
// item counter, ~1.2 million atomics per iteration at 200 uneven slices,
// cost 14 ms where the pixels take 1.6 ms).
__global__ void __launch_bounds__(kPixBlock)
k_update_batch(const BatchSliceDev *__restrict__ d, BatchQueues q, int it) {
  const int *start = q.start[2];
  const int total = start[q.n];
  for (;;) {
    const int item = batch_next_item(q.counters + 2);
    if (item >= total) break;
    const int k = batch_find(start, q.n, item);
    const BatchSliceDev &sd = d[__builtin_amdgcn_readfirstlane(q.order[2][k])];
    if (it >= sd.iters) continue;
    const int64_t NN = (int64_t)sd.g.N * sd.g.N;
    const int64_t j0 = (int64_t)(item - start[k]) * kPixBlock * kBatchUpdateBlocks + threadIdx.x;
#pragma unroll 4
    for (int u = 0; u < kBatchUpdateBlocks; ++u) {
      const int64_t j = j0 + (int64_t)u * kPixBlock;
      if (j < NN) {
        float xv = sd.x[j];
        if (sd.alg == 0) xv += sd.z[j] / sd.den[j];
        else xv *= sd.z[j] / sd.den[j];
        sd.x[j] = xv;
      }
    }
  }
}

// ------------------------------------------------- reference / debugging --

// Whole-ray scatter with global atomics (z must be zeroed): the plain
// ray-driven adjoint, kept as an independent check of the tile kernel.
template <bool kExact>
__global__ void __launch_bounds__(kRayBlock)
k_adjoint_atomic(GridInfo g, const AngleInfo *__restrict__ ang,
                 const RayInfo *__restrict__ rays, int P, int S, int mode,
                 const float *__restrict__ r, float *__restrict__ z) {
  const int64_t t = (int64_t)blockIdx.x * kRayBlock + threadIdx.x;
  const int C = g.C;
  if (t >= (int64_t)P * C) return;
  const int p = (int)(t / C);
  const int s = blockIdx.y;
  const unsigned NN = (unsigned)g.N * (unsigned)g.N;
  float w = 1.f;
  if (mode == kBpSino) {
    w = r[t * S + s];  // [P][C][S]
    if (w == 0.f) return;
  }
  float *zs = z + (int64_t)s * NN;
  traverse_full<kExact>(g, rays[t], ang[p].quadrant, [&](int ix, int iy, float l, float) {
    const unsigned idx = (unsigned)(ix + iy * g.N);
    if (idx < NN) atomic_add_f32(zs + idx, mode == kBpCount ? 1.0f : (mode == kBpOnes ? l : l * w));
  });
}

template <bool kExact>
__global__ void k_dump_rays(GridInfo g, const AngleInfo *__restrict__ ang,
                            const RayInfo *__restrict__ rays, int n,
                            const int *__restrict__ proj, const int *__restrict__ col,
                            int max_seg, int *__restrict__ counts, int *__restrict__ idx,
                            float *__restrict__ len, float *__restrict__ len2) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  int k = 0;
  const int64_t base = (int64_t)t * max_seg;
  const int64_t ray = (int64_t)proj[t] * g.C + col[t];
  const int cnt = traverse_full<kExact>(g, rays[ray], ang[proj[t]].quadrant,
                                        [&](int ix, int iy, float l, float l2) {
                                          if (k < max_seg) {
                                            idx[base + k] = ix + iy * g.N;
                                            len[base + k] = l;
                                            len2[base + k] = l2;
                                          }
                                          ++k;
                                        });
  counts[t] = cnt;
}

// Per-ray sums over all segments, in the walk order: len_sum = sum len
// (row sums of A) and len2_sum = sum len^2 (the SIRT normaliser a2 of
// sirt.cc:47-50, accumulated from the squared lengths as there).  Output
// [P][C]; either pointer may be null.
template <bool kExact>
__global__ void __launch_bounds__(kRayBlock)
k_ray_sums(GridInfo g, const AngleInfo *__restrict__ ang, const RayInfo *__restrict__ rays,
           int P, float *__restrict__ len_sum, float *__restrict__ len2_sum) {
  const int64_t t = (int64_t)blockIdx.x * kRayBlock + threadIdx.x;
  if (t >= (int64_t)P * g.C) return;
  const int p = (int)(t / g.C);
  float a1 = 0.f, a2 = 0.f;
  traverse_full<kExact>(g, rays[t], ang[p].quadrant, [&](int, int, float l, float l2) {
    a1 += l;
    a2 += l2;
  });
  if (len_sum) len_sum[t] = a1;
  if (len2_sum) len2_sum[t] = a2;
}

__global__ void k_check_finite(const float *__restrict__ v, int64_t n,
                               int *__restrict__ flag) {
  int64_t i = (int64_t)blockIdx.x * kPixBlock + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * kPixBlock;
  int bad = 0;
  for (; i < n; i += stride) bad |= !__builtin_isfinite(v[i]);
  if (bad) atomicOr(flag, 1);
}

inline unsigned blocks_for(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

// ------------------------------------------------ launch-shape dispatch --

template <int SB, bool E, int LPR, bool kWide>
hipError_t fwd_mode(int mode, const Geometry &g, const RayInfo *rays, int ba_log2,
                    const float *xb, const float *sino, float *out, unsigned *maxw,
                    hipStream_t st) {
  const int bc = (64 / LPR) >> ba_log2, ba = 1 << ba_log2;
  if (bc < 1) return hipErrorInvalidValue;
  const int64_t bundles = (int64_t)((g.P + ba - 1) / ba) * ((g.C + bc - 1) / bc);
  dim3 grid(blocks_for(bundles, kRayBlock / 64), (g.S + SB - 1) / SB), block(kRayBlock);
  if (mode == kFwdY)
    hipLaunchKernelGGL((k_forward<SB, kFwdY, E, LPR, kWide>), grid, block, 0, st, g.grid,
                       g.d_ang, rays, g.P, g.S, ba_log2, xb, sino, out, maxw);
  else if (mode == kFwdSIRT)
    hipLaunchKernelGGL((k_forward<SB, kFwdSIRT, E, LPR, kWide>), grid, block, 0, st, g.grid,
                       g.d_ang, rays, g.P, g.S, ba_log2, xb, sino, out, maxw);
  else
    hipLaunchKernelGGL((k_forward<SB, kFwdEM, E, LPR, kWide>), grid, block, 0, st, g.grid,
                       g.d_ang, rays, g.P, g.S, ba_log2, xb, sino, out, maxw);
  return hipGetLastError();
}

template <int SB, int LPR>
hipError_t fwd_exact(bool exact, int mode, const Geometry &g, const RayInfo *rays, int ba_log2,
                     const float *xb, const float *sino, float *out, unsigned *maxw,
                     hipStream_t st) {
  if (wide_image(g.N, SB)) {
    if constexpr (SB == 1 && LPR == 1)
      return exact ? fwd_mode<1, true, 1, true>(mode, g, rays, ba_log2, xb, sino, out, maxw, st)
                   : fwd_mode<1, false, 1, true>(mode, g, rays, ba_log2, xb, sino, out, maxw, st);
    return hipErrorInvalidValue;
  }
  return exact
             ? fwd_mode<SB, true, LPR, false>(mode, g, rays, ba_log2, xb, sino, out, maxw, st)
             : fwd_mode<SB, false, LPR, false>(mode, g, rays, ba_log2, xb, sino, out, maxw, st);
}

constexpr size_t kLdsBytes = 160 * 1024;

template <int TW, int TH, int SB, int MODE, bool E, int BLK>
hipError_t bp_launch(TileArgs a, int nbatch, hipStream_t st) {
  const int N = a.g.N;
  const int tiles = ((N + TW - 1) / TW) * ((N + TH - 1) / TH);
  size_t lds = (size_t)bp_acc_words<TW, TH, SB, MODE>() * sizeof(BpWord<MODE>);
  // stage the per-angle column counts in LDS when they fit
  a.count_lds = (lds + (size_t)a.P * sizeof(int) <= kLdsBytes / 2) ? 1 : 0;
  if (a.count_lds) lds += (size_t)a.P * sizeof(int);
  auto kern = k_bp_tile<TW, TH, SB, MODE, E, BLK>;
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute((const void *)kern,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kern, dim3(tiles, nbatch), dim3(BLK), lds, st, a);
  return hipGetLastError();
}

// Lanes of a tile's workgroup: the fewest of 256, 512 and 1024 that leave a CU
// with 24 wavefronts (or what the vector registers allow), counting the
// workgroups there are and those whose accumulators fit its LDS; 1024 only
// where tiles are scarce, since a workgroup ends with its slowest lane.  One
// launch with 256 / 512 / 1024 lanes (us):
//   1 slice, 16x16, 256^2, 180 angles      92 /    53 /    41
//   1 slice, 32x32, 1024^2, 720 angles   1415 /  1229 /  1412
//   1 slice, 64x64, 2048^2, 1500 angles  9233 /  8173 /  9309
//   5 slices, 32x32x8, 1024^2, 720       2800 /  1810 /  2189
//   12 slices, 16x16x16, 2048^2, 1500   24855 / 29672 / 37040
int tile_block(int N, int P, int TW, int TH, int SB, int nbatch) {
  const int64_t tiles = (int64_t)((N + TW - 1) / TW) * ((N + TH - 1) / TH) * nbatch;
  const double per_cu = tiles / 256.0;
  if (per_cu <= 1.0) return 1024;  // a CU holds one such workgroup
  // a launch holds fewer than 2^32 lanes (8x8 tiles from 23171^2 on)
  if (tiles / nbatch * 512 >= (int64_t(1) << 32)) return 256;
  const size_t lds = (size_t)TH * (TW + 1) * 4 * (SB + (SB > 1 ? 1 : 0)) + (size_t)P * sizeof(int);
  const int waves = SB <= 8 ? 28 : (SB <= 16 ? 20 : 12);  // by vector registers
  const int want = waves < 24 ? waves : 24;
  const double resident = std::fmin(per_cu, std::fmin((double)(kLdsBytes / lds), waves / 4.0));
  return resident * 4 >= want ? 256 : 512;
}

template <int SB, bool E>
hipError_t bp_split_launch(const TileArgs &a, int nbatch, hipStream_t st) {
  constexpr int BLK = kTileBlock;
  const int tiles = ((a.g.N + 15) / 16) * ((a.g.N + 15) / 16);
  constexpr size_t lds = (size_t)bp_acc_words<16, 16, SB, kBpSino>() * sizeof(unsigned);
  static_assert(lds <= 65536, "no attribute needed");
  hipLaunchKernelGGL((k_bp_tile_split<16, 16, SB, E, BLK>), dim3(tiles, nbatch, a.split.n),
                     dim3(BLK), lds, st, a);
  return hipGetLastError();
}

template <int TW, int TH, int SB>
hipError_t bp_mode(int mode, bool exact, const TileArgs &a, int nbatch, hipStream_t st) {
  if constexpr (TW == 16 && TH == 16)
    if (mode == kBpSino && a.split.n > 1)
      return exact ? bp_split_launch<SB, true>(a, nbatch, st)
                   : bp_split_launch<SB, false>(a, nbatch, st);
  if (mode == kBpSino) {
    const int blk = tile_block(a.g.N, a.P, TW, TH, SB, nbatch);
    if constexpr (SB <= 16)
      if (blk == 1024)
        return exact ? bp_launch<TW, TH, SB, kBpSino, true, 1024>(a, nbatch, st)
                     : bp_launch<TW, TH, SB, kBpSino, false, 1024>(a, nbatch, st);
    if (blk >= 512)
      return exact ? bp_launch<TW, TH, SB, kBpSino, true, 512>(a, nbatch, st)
                   : bp_launch<TW, TH, SB, kBpSino, false, 512>(a, nbatch, st);
    return exact ? bp_launch<TW, TH, SB, kBpSino, true, 256>(a, nbatch, st)
                 : bp_launch<TW, TH, SB, kBpSino, false, 256>(a, nbatch, st);
  }
  if (mode == kBpOnes)
    return exact ? bp_launch<TW, TH, 1, kBpOnes, true, 256>(a, 1, st)
                 : bp_launch<TW, TH, 1, kBpOnes, false, 256>(a, 1, st);
  return bp_launch<TW, TH, 1, kBpCount, true, 256>(a, 1, st);
}

}  // namespace

// ------------------------------------------------------------ launchers --

int tile_count_bound(float sinq, float cosq, int TW, int TH) {
  // columns in an interval of length TW|sin| + TH|cos| + 2 kColumnMargin
  // (plus rounding of the float projections, far below the 2 x 0.05 pixel
  // that kCountMargin adds): at most floor(len) + 1.
  // At most ceil(sqrt(TW^2 + TH^2)) + 4, the column ranks bp_tile_loop
  // enumerates for one-slice tiles (ensure_count checks it).
  const double len =
      TW * std::fabs((double)sinq) + TH * std::fabs((double)cosq) + 2.0 * kCountMargin;
  return (int)std::floor(len) + 1;
}

hipError_t launch_ray_info(const Geometry &g, RayInfo *rays, unsigned long long *counts,
                           hipStream_t st) {
  const int64_t n = g.rays_per_slice();
  hipLaunchKernelGGL(k_ray_info, dim3(blocks_for(n, kRayBlock)), dim3(kRayBlock), 0, st,
                     g.grid, g.d_ang, g.d_yi, g.P, counts, rays);
  return hipGetLastError();
}

hipError_t launch_forward(const Geometry &g, const RayInfo *rays, int sb, int bundle_angles,
                          int lanes_per_ray, int mode, bool exact, const float *xb,
                          const float *sino, float *out, unsigned *maxw, hipStream_t st) {
  int ba_log2 = 0;
  while ((1 << ba_log2) < bundle_angles && ba_log2 < 6) ++ba_log2;
  if ((1 << ba_log2) != bundle_angles) return hipErrorInvalidValue;
#define TRACE_FWD_CASE(SB_, LPR_)                                                    \
  if (sb == SB_ && lanes_per_ray == LPR_)                                            \
    return fwd_exact<SB_, LPR_>(exact, mode, g, rays, ba_log2, xb, sino, out, maxw, st);
  TRACE_FWD_SHAPES(TRACE_FWD_CASE)
#undef TRACE_FWD_CASE
  return hipErrorInvalidValue;
}

int tile_splits(const Geometry &g, const TileShape &ts, int n_slices, int64_t whole_rays) {
  if (ts.tw != 16 || ts.th != 16) return 1;
  const int64_t items = (int64_t)((g.N + 15) / 16) * ((g.N + 15) / 16) * ((n_slices + ts.sb - 1) / ts.sb);
  const int64_t pairs = (int64_t)g.P * 22;  // (angle, column) pairs of a tile
  // one workgroup has two pairs a lane from 2048 on (1024 lanes; 512 at 32
  // slices), which pays for adding the parts, later where these are many words
  // (8 and 16 slices) or wait for each other on busy CUs (many items).  One
  // workgroup / several (us) at 94, 110, 125 and 145 angles:
  //   1 slice    90^2   24 / 22   26 / 23   31 / 23   33 / 24
  //             176^2   25 / 26   27 / 28   31 / 29   34 / 29
  //   4 slices  176^2   36 / 39   41 / 39   42 / 40   50 / 42
  //   8 slices   90^2   38 / 41   43 / 42   45 / 45   53 / 50
  //             176^2   39 / 46   44 / 47   46 / 48   54 / 49
  //  16 slices   90^2   52 / 55   59 / 56   62 / 56   73 / 57
  //             176^2   53 / 62   60 / 63   63 / 66   74 / 68
  //  32 slices  176^2   78 / 76   87 / 85   93 / 88  105 / 100
  // Where many rays are walked whole (angles past a half turn), a pair is worth
  // the more: 8 slices 125^2 at 108 angles over a full turn 73 / 62.
  const bool long_walks = whole_rays * 8 > g.rays_per_slice();
  const int64_t least = long_walks                  ? 2048
                        : ts.sb == 8 || ts.sb == 16 ? 2100 + 8 * items
                        : ts.sb <= 4 && items > 74  ? 1600 + 6 * items
                                                    : 2048;
  if (items > 128 || pairs < least) return 1;
  // up to four workgroups of 256 lanes a CU, a pair for every lane, and at most
  // 32768 words for the last one to add up
  int64_t n = 1024 / items;
  const int64_t words = 32768 / ((ts.sb + 1) * TilePitch<16, 16>::kPlane);
  n = n < pairs / kTileBlock ? n : pairs / kTileBlock;
  n = n < words ? n : words;
  if (n < 2) return 1;
  const int64_t per = (g.P + n - 1) / n;
  return (int)((g.P + per - 1) / per);
}

size_t tile_split_words(const Geometry &g, const TileShape &ts, int n_slices, int splits) {
  const size_t items = (size_t)((g.N + 15) / 16) * ((g.N + 15) / 16) * ((n_slices + ts.sb - 1) / ts.sb);
  return items * splits * (ts.sb + 1) * TilePitch<16, 16>::kPlane;
}

hipError_t launch_backproject(const Geometry &g, const RayInfo *rays, const int *count,
                              const TileShape &ts, int mode, bool exact, const float *w,
                              const unsigned *maxw, float maxlen, float denmax, float *z,
                              bool wraps, const TileSplit &split, int s0, int n,
                              hipStream_t st) {
  TileArgs a;
  a.split = split;
  a.wraps = wraps ? 1 : 0;
  a.maxw = maxw ? maxw + s0 : nullptr;
  a.maxlen = maxlen;
  a.denmax = denmax;
  a.g = g.grid;
  a.ang = g.d_ang;
  a.rays = rays;
  a.count = count;
  a.P = g.P;
  a.S = g.S;
  a.n = n;
  a.yi0 = g.yi0;
  a.w = w ? w + s0 : nullptr;
  a.z = z + (int64_t)s0 * g.NN();
  const int nb = (n + ts.sb - 1) / ts.sb;
#define TRACE_BP_CASE(TW_, TH_, SB_)                              \
  if (ts.tw == TW_ && ts.th == TH_ && ts.sb == SB_)               \
    return bp_mode<TW_, TH_, SB_>(mode, exact, a, nb, st);
  TRACE_BP_SHAPES(TRACE_BP_CASE)
#undef TRACE_BP_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_pack(const float *src, int nsrc, int off, float fill, int64_t NN, int nslots,
                       int sb, float *xb, hipStream_t st) {
  const int nb = (nslots + sb - 1) / sb;
  dim3 grid(blocks_for(NN, kPixBlock), nb), block(kPixBlock);
  switch (sb) {
    case 1: hipLaunchKernelGGL(k_pack<1>, grid, block, 0, st, src, nsrc, off, fill, NN, nslots, xb); break;
    case 2: hipLaunchKernelGGL(k_pack<2>, grid, block, 0, st, src, nsrc, off, fill, NN, nslots, xb); break;
    case 4: hipLaunchKernelGGL(k_pack<4>, grid, block, 0, st, src, nsrc, off, fill, NN, nslots, xb); break;
    case 8: hipLaunchKernelGGL(k_pack<8>, grid, block, 0, st, src, nsrc, off, fill, NN, nslots, xb); break;
    case 16: hipLaunchKernelGGL(k_pack<16>, grid, block, 0, st, src, nsrc, off, fill, NN, nslots, xb); break;
    case 32: hipLaunchKernelGGL(k_pack<32>, grid, block, 0, st, src, nsrc, off, fill, NN, nslots, xb); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// Slices per thread of the updates: the slot batch, or 4 of it where that
// leaves too few workgroups, since a thread takes its slices one after the other
// (APMLR some 10 divisions and a square root each: below 2048 workgroups, SIRT
// and MLEM one division: below 512).  All / 4 slices (us): APMLR 14 slices 82^2
// 58 / 18, 9 slices 511^2 59 / 39; PML 20 slices 151^2 45 / 14; SIRT 33 slices
// 125^2 15 / 7; MLEM 7 slices 548^2 8 / 10.  Where the wavefronts are there
// anyway whole lines of the copy are written.
static bool update_split(int64_t NN, int sb, int slots, int blocks) {
  return sb > 4 && (int64_t)blocks_for(NN, kPixBlock) * ((slots + sb - 1) / sb) < blocks;
}

hipError_t launch_update_em(bool sirt, float *x, const float *z, const float *den, int S,
                            int64_t NN, int sb, float *xb, unsigned *maxw, hipStream_t st) {
  const int nslots = (S + sb - 1) / sb * sb;
  const int vb = update_split(NN, sb, nslots, 512) ? 4 : sb;
  const dim3 grid(blocks_for(NN, kPixBlock), nslots / vb), block(kPixBlock);
#define TRACE_UPD_CASE(SB_, VB_)                                                            \
  if (sb == SB_ && vb == VB_) {                                                             \
    if (sirt)                                                                               \
      hipLaunchKernelGGL((k_update_em<SB_, VB_, true>), grid, block, 0, st, x, z, den, S,   \
                         NN, xb, maxw);                                                     \
    else                                                                                    \
      hipLaunchKernelGGL((k_update_em<SB_, VB_, false>), grid, block, 0, st, x, z, den, S,  \
                         NN, xb, maxw);                                                     \
    return hipGetLastError();                                                               \
  }
  TRACE_UPDATE_SHAPES(TRACE_UPD_CASE)
#undef TRACE_UPD_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_fill(float *p, int64_t n, float v, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill, dim3(blocks_for(n, kPixBlock)), dim3(kPixBlock), 0, st, p, n, v);
  return hipGetLastError();
}

hipError_t launch_update_pml(const float *x, float *xn, const float *z, const float *den,
                             int S, int N, float beta, bool num_direct, int sb, int nslots,
                             float *xb, unsigned *maxw, hipStream_t st) {
  const unsigned bx = blocks_for((int64_t)N * N, kPixBlock);
  const int vb = update_split((int64_t)N * N, sb, nslots, 2048) ? 4 : sb;
  const dim3 grid(bx, nslots / vb);
#define TRACE_PML_CASE(SB_, VB_)                                                           \
  if (sb == SB_ && vb == VB_) {                                                            \
    hipLaunchKernelGGL((k_update_pml<SB_, VB_>), grid, dim3(kPixBlock), 0, st, x, xn, z,   \
                       den, S, N, beta, num_direct ? 1 : 0, xb, maxw);                     \
    return hipGetLastError();                                                              \
  }
  TRACE_UPDATE_SHAPES(TRACE_PML_CASE)
#undef TRACE_PML_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_update_apmlr(const float *xpad, float *xnpad, const float *z,
                               const float *den, int S, int N, const RegParams &p,
                               const StencilWeights &w, int compat, bool num_direct,
                               int sb, int nslots, float *xb, unsigned *maxw, hipStream_t st) {
  // slots: those of the copy and every real slice's
  const int off = compat ? 0 : 1;
  const int need = (nslots > S + 1 - off) ? nslots : S + 1 - off;
  const int vb = update_split((int64_t)N * N, sb, need, 2048) ? 4 : sb;
  const dim3 grid(blocks_for((int64_t)N * N, kPixBlock), (need + vb - 1) / vb);
  ApmlrArgs a{w, p, compat, nslots, num_direct ? 1 : 0};
#define TRACE_APMLR_CASE(SB_, VB_)                                                         \
  if (sb == SB_ && vb == VB_) {                                                            \
    hipLaunchKernelGGL((k_update_apmlr<SB_, VB_>), grid, dim3(kPixBlock), 0, st, xpad,     \
                       xnpad, z, den, S, N, a, xb, maxw);                                  \
    return hipGetLastError();                                                              \
  }
  TRACE_UPDATE_SHAPES(TRACE_APMLR_CASE)
#undef TRACE_APMLR_CASE
  return hipErrorInvalidValue;
}

hipError_t launch_batch_reset(const BatchQueues &q, hipStream_t st) {
  const int n = q.n > 3 ? q.n : 3;
  hipLaunchKernelGGL(k_batch_reset, dim3((n + 255) / 256), dim3(256), 0, st, q.counters,
                     q.maxw_all, q.n);
  return hipGetLastError();
}

hipError_t launch_batch_forward(const BatchSliceDev *d, const BatchQueues &q, int it,
                                int bundle_angles, bool exact, int grid, hipStream_t st) {
  int ba_log2 = 0;
  while ((1 << ba_log2) < bundle_angles && ba_log2 < 6) ++ba_log2;
  if ((1 << ba_log2) != bundle_angles || grid <= 0) return hipErrorInvalidValue;
  if (exact)
    hipLaunchKernelGGL(k_forward_batch<true>, dim3(grid), dim3(kRayBlock), 0, st, d, q, it,
                       ba_log2);
  else
    hipLaunchKernelGGL(k_forward_batch<false>, dim3(grid), dim3(kRayBlock), 0, st, d, q, it,
                       ba_log2);
  return hipGetLastError();
}

hipError_t launch_batch_backproject(const BatchSliceDev *d, const BatchQueues &q, int it,
                                    int tw, int th, bool exact, int grid, size_t lds,
                                    hipStream_t st) {
  if (grid <= 0) return hipErrorInvalidValue;
#define TRACE_BATCH_BP(TW_, TH_)                                                             \
  if (tw == TW_ && th == TH_) {                                                              \
    if (exact)                                                                               \
      hipLaunchKernelGGL((k_bp_batch<TW_, TH_, true>), dim3(grid), dim3(kTileBlock), lds, st, \
                         d, q, it);                                                          \
    else                                                                                     \
      hipLaunchKernelGGL((k_bp_batch<TW_, TH_, false>), dim3(grid), dim3(kTileBlock), lds,    \
                         st, d, q, it);                                                      \
    return hipGetLastError();                                                                \
  }
  TRACE_BATCH_TILES(TRACE_BATCH_BP)
#undef TRACE_BATCH_BP
  return hipErrorInvalidValue;
}

hipError_t launch_batch_update(const BatchSliceDev *d, const BatchQueues &q, int it, int grid,
                               hipStream_t st) {
  if (grid <= 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_update_batch, dim3(grid), dim3(kPixBlock), 0, st, d, q, it);
  return hipGetLastError();
}

bool batch_tile_supported(int tw, int th) {
#define TRACE_BATCH_MATCH(TW_, TH_) \
  if (tw == TW_ && th == TH_) return true;
  TRACE_BATCH_TILES(TRACE_BATCH_MATCH)
#undef TRACE_BATCH_MATCH
  return false;
}

int batch_blocks_per_cu(int phase, int tw, int th, bool exact, size_t lds) {
  int nb = 0;
  hipError_t e = hipErrorInvalidValue;
  if (phase == 0) {
    e = exact ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_forward_batch<true>,
                                                             kRayBlock, 0)
              : hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_forward_batch<false>,
                                                             kRayBlock, 0);
  } else if (phase == 2) {
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_update_batch, kPixBlock, 0);
  } else {
#define TRACE_BATCH_OCC(TW_, TH_)                                                            \
  if (tw == TW_ && th == TH_)                                                                \
    e = exact ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_bp_batch<TW_, TH_, true>, \
                                                             kTileBlock, lds)                \
              : hipOccupancyMaxActiveBlocksPerMultiprocessor(                                \
                    &nb, k_bp_batch<TW_, TH_, false>, kTileBlock, lds);
    TRACE_BATCH_TILES(TRACE_BATCH_OCC)
#undef TRACE_BATCH_OCC
  }
  return e == hipSuccess ? nb : 0;
}

hipError_t launch_adjoint_atomic(const Geometry &g, const RayInfo *rays, int mode, bool exact,
                                 const float *r, float *z, int nslices, hipStream_t st) {
  const int64_t n = g.rays_per_slice();
  dim3 grid(blocks_for(n, kRayBlock), nslices), block(kRayBlock);
  if (exact)
    hipLaunchKernelGGL(k_adjoint_atomic<true>, grid, block, 0, st, g.grid, g.d_ang, rays, g.P,
                       g.S, mode, r, z);
  else
    hipLaunchKernelGGL(k_adjoint_atomic<false>, grid, block, 0, st, g.grid, g.d_ang, rays, g.P,
                       g.S, mode, r, z);
  return hipGetLastError();
}

hipError_t launch_dump_rays(const Geometry &g, const RayInfo *rays, int n, const int *proj,
                            const int *col, int max_seg, int *counts, int *idx, float *len,
                            float *len2, hipStream_t st, bool exact) {
  if (n <= 0) return hipSuccess;
  if (exact)
    hipLaunchKernelGGL(k_dump_rays<true>, dim3(blocks_for(n, 64)), dim3(64), 0, st, g.grid,
                       g.d_ang, rays, n, proj, col, max_seg, counts, idx, len, len2);
  else
    hipLaunchKernelGGL(k_dump_rays<false>, dim3(blocks_for(n, 64)), dim3(64), 0, st, g.grid,
                       g.d_ang, rays, n, proj, col, max_seg, counts, idx, len, len2);
  return hipGetLastError();
}

hipError_t launch_ray_sums(const Geometry &g, const RayInfo *rays, bool exact, float *len_sum,
                           float *len2_sum, hipStream_t st) {
  const int64_t n = g.rays_per_slice();
  if (exact)
    hipLaunchKernelGGL(k_ray_sums<true>, dim3(blocks_for(n, kRayBlock)), dim3(kRayBlock), 0, st,
                       g.grid, g.d_ang, rays, g.P, len_sum, len2_sum);
  else
    hipLaunchKernelGGL(k_ray_sums<false>, dim3(blocks_for(n, kRayBlock)), dim3(kRayBlock), 0, st,
                       g.grid, g.d_ang, rays, g.P, len_sum, len2_sum);
  return hipGetLastError();
}

hipError_t launch_to_pcs(const float *r, int P, int S, int C, float *w, unsigned *maxw,
                         hipStream_t st) {
  const int64_t blocks = (int64_t)P * ((C + 63) / 64);
  hipLaunchKernelGGL(k_to_pcs,
                     dim3((unsigned)(blocks < 2048 ? blocks : 2048), (S + kTransS - 1) / kTransS),
                     dim3(256), 0, st, r, P, S, C, w, maxw);
  return hipGetLastError();
}

hipError_t launch_absmax_slices(const float *w, int P, int S, int C, unsigned *maxw,
                                hipStream_t st) {
  int64_t n = (int64_t)P * C;
  unsigned bx = blocks_for(n, 4 * kPixBlock);
  if (bx > 512) bx = 512;
  hipLaunchKernelGGL(k_absmax_slices, dim3(bx, S), dim3(kPixBlock), 0, st, w, P, S, C, maxw);
  return hipGetLastError();
}

hipError_t launch_check_finite(const float *v, int64_t n, int *flag, hipStream_t st) {
  unsigned blocks = blocks_for(n, kPixBlock);
  if (blocks > 4096) blocks = 4096;
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_check_finite, dim3(blocks), dim3(kPixBlock), 0, st, v, n, flag);
  return hipGetLastError();
}

}  // namespace trace_hip
