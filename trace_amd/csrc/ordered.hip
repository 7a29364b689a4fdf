// ordered.hip -- backprojection summed in the reference's order.
//
// The reference accumulates each pixel's backprojected sums in float, one
// segment at a time, in the order its one-thread engine meets the rays:
// projections ascending, detector columns ascending, segments along the ray
// (rows of NextMirroredRegion, data_region_base.h:98-111; the per-segment
// updates of UpdateReconReplica):
//
//   den_j += len                      sirt.cc:62, mlem.cc:57, pml.cc:244
//   num_j += len * upd                sirt.cc:61, mlem.cc:56
//   num_j -= (x_j * len) * upd        pml.cc:243, apmlr.cc:1024
//
// A float sum depends on its order.  For PML and APMLR it matters: the
// closed-form update (pml.cc:18-20) evaluates -G + sqrt(G^2 - 8 num F) with
// G ~ den ~ P, which cancels, so one ulp of den or num in G^2 - 8 num F
// moves the updated pixel by up to ~1e-4 relative.  The tile backprojector
// (kernels.hip) sums in fixed point, exactly but in no particular order;
// this one reproduces the reference's float sums bit for bit.
//
// Gather form: each thread owns a strip of PW x PH pixels and loops over
// the projections in order; per projection it walks the columns whose ray
// can touch the strip in ascending order (tile_columns), each over the
// window of the ray around the strip (traverse_window, the same walk the
// tile kernels use), and adds the segments falling in the strip to its
// register accumulators.  Every pixel's terms therefore arrive in the
// reference's (projection, column, segment) order.  No atomics, no LDS.
//
// Wrapped segments (ix == N: the reference's truncation sends them to pixel
// 0 of the next row, trace_utils.cc:177-185) belong to strips at column 0.
// Such strips walk the flagged rays (kRayWraps) crossing the strip left of
// the right edge whole, so that their segments keep the ray's order.
//
// Tile form (k_bp_ordered_tile, the default where it applies): a wavefront
// owns an 8 x 8 tile and takes the projections four at a time.  Its 64
// lanes first walk the four projections' columns through the tile at once
// (one (projection, column) pair per lane, as the LDS tile backprojector
// does) and drop every segment's length into an LDS slot keyed by (pixel,
// projection, column modulo 3, segment number of that ray in that pixel);
// then each lane sums its own pixel's slots in (projection, column, segment)
// order.  A pixel sees at most three candidate columns per projection (its
// projected width is at most sqrt 2 plus twice the 0.45-pixel margin), so
// the column modulo 3 tells them apart, and a ray puts at most two segments
// in one pixel, one after the other, on the geometries measured (two where
// it grazes a corner); a geometry that would need more sets a flag when den
// is computed.  Geometries with rays on grid lines need more, and have
// wrapped segments: a variant of the shared form below serves them where it is
// the faster (ordered_grid_pays), and the per-pixel form elsewhere and what
// overflows there too.
//
// The walks bound the one-slice form, the sums the deeper ones.  Filing a
// segment waits for nothing: its slot is the lane's own (the ray's column
// modulo 3, and whether the segment before it fell in the same pixel), and
// its presence is counted without reading the count back.  With the slot
// from a table of first columns and the number from the count, two LDS round
// trips a segment, the column sums of 2048^2 / 1500 took 45.3 ms instead of 37.1.
#include <hip/hip_runtime.h>

#include <cmath>

#include "internal.h"

#pragma clang fp contract(off)

namespace trace_hip {

namespace {

constexpr int kOrdBlock = 256;
constexpr int kOrdStrips = 16;  // a block is 16 x 16 strips

struct OrdArgs {
  GridInfo g;
  const AngleInfo *ang;
  const RayInfo *rays;
  int P, S;         // S: slices of a row of w
  int n;            // slices from w, xb and out on
  float yi0;
  const float *w;   // [P][C][S] per-ray weights (kOrdNum, kOrdEM)
  const float *xb;  // [S/xsb][N*N][xsb] image the ray pass read (kOrdNum)
  int xsb;          // slices per slot batch of xb
  float *out;       // kOrdDen: [N][N]; kOrdNum, kOrdEM: [S][N][N]
  int wraps;        // some ray has a segment with ix == N
};

template <int PW, int PH, int SB, int MODE, bool kExact>
__global__ void __launch_bounds__(kOrdBlock)
k_bp_ordered(OrdArgs a) {
  constexpr int NP = PW * PH;
  const int N = a.g.N, C = a.g.C;
  const int sxn = (N + PW - 1) / PW, syn = (N + PH - 1) / PH;
  const int bxn = (sxn + kOrdStrips - 1) / kOrdStrips;
  const int sx = (int)(blockIdx.x % bxn) * kOrdStrips + (threadIdx.x % kOrdStrips);
  const int sy = (int)(blockIdx.x / bxn) * kOrdStrips + (threadIdx.x / kOrdStrips);
  if (sx >= sxn || sy >= syn) return;  // no barrier in this kernel
  const int tx0 = sx * PW, ty0 = sy * PH;
  const int tx1 = min(tx0 + PW, N), ty1 = min(ty0 + PH, N);
  const int b = blockIdx.y;
  const int64_t NN = (int64_t)N * N;

  float acc[NP][SB];
  float xv[NP][SB];
#pragma unroll
  for (int i = 0; i < NP; ++i)
#pragma unroll
    for (int q = 0; q < SB; ++q) acc[i][q] = 0.f, xv[i][q] = 0.f;
  if (MODE == kOrdNum) {
    // x of the ray pass, slots b*SB .. b*SB+SB-1 (SB divides xsb)
    const int s0 = b * SB;
    const int xb_b = s0 / a.xsb, xb_q = s0 % a.xsb;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int px = tx0 + i % PW, py = ty0 + i / PW;
      if (px < N && py < N) {
        const float *src = a.xb + ((int64_t)xb_b * NN + (int64_t)py * N + px) * a.xsb + xb_q;
#pragma unroll
        for (int q = 0; q < SB; ++q) xv[i][q] = src[q];
      }
    }
  }
  const float x0 = grid_line(N, tx0), x1 = grid_line(N, tx1);
  const float y0 = grid_line(N, ty0), y1 = grid_line(N, ty1);
  // strip just left of the right edge, rows ty0-1 .. ty1: the rays whose
  // wrapped segments can land in a column-0 strip
  const bool edge = a.wraps && tx0 == 0;
  const float ex0 = grid_line(N, N - 1), ex1 = grid_line(N, N);
  const float ey0 = grid_line(N, ty0 - 1), ey1 = y1;

  for (int p = 0; p < a.P; ++p) {
    const AngleInfo ang = a.ang[p];
    int cmin, cmax;
    tile_columns(ang, x0, x1, y0, y1, a.yi0, cmin, cmax);
    int emin = 1, emax = 0;
    if (edge) tile_columns(ang, ex0, ex1, ey0, ey1, a.yi0, emin, emax);
    const int lo = max(0, edge ? min(cmin, emin) : cmin);
    const int hi = min(C - 1, edge ? max(cmax, emax) : cmax);
    for (int c = lo; c <= hi; ++c) {
      const bool in_main = (c >= cmin && c <= cmax);
      const bool in_erange = edge && c >= emin && c <= emax;
      if (!in_main && !in_erange) {
        // c lies in the gap between the two ranges: go to the upper one
        c = (c > cmax ? emin : cmin) - 1;
        continue;
      }
      const int64_t t = (int64_t)p * C + c;
      const RayInfo ray = a.rays[t];
      const bool in_edge = in_erange && (ray.alo & kRayWraps);
      if (!in_main && !in_edge) continue;
      float wv[SB];
      if (MODE != kOrdDen) {
        const float *wr = a.w + t * a.S + b * SB;
#pragma unroll
        for (int q = 0; q < SB; ++q) wv[q] = (b * SB + q < a.n) ? wr[q] : 0.f;
      }
      auto visit = [&](int ix, int iy, float l, float) {
        const bool wrap = (ix == N);
        if (wrap && !in_edge) return;
        ix = wrap ? 0 : ix;
        iy = wrap ? iy + 1 : iy;
        const unsigned lx = (unsigned)(ix - tx0), ly = (unsigned)(iy - ty0);
        if (lx < (unsigned)(tx1 - tx0) && ly < (unsigned)(ty1 - ty0)) {
          const int pix = (int)(ly * PW + lx);
#pragma unroll
          for (int i = 0; i < NP; ++i) {
            if (NP == 1 || pix == i) {
#pragma unroll
              for (int q = 0; q < SB; ++q) {
                if (MODE == kOrdDen)
                  acc[i][q] = acc[i][q] + l;
                else if (MODE == kOrdEM)
                  acc[i][q] = acc[i][q] + l * wv[q];
                else
                  acc[i][q] = acc[i][q] - (xv[i][q] * l) * wv[q];
              }
            }
          }
        }
      };
      if (in_edge)
        traverse_full<kExact>(a.g, ray, ang.quadrant, visit);
      else
        traverse_window<kExact, true>(a.g, ray, ang.quadrant, tx0, tx1, ty0, ty1, visit);
    }
  }
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int px = tx0 + i % PW, py = ty0 + i / PW;
    if (px >= N || py >= N) continue;
    const int64_t j = (int64_t)py * N + px;
#pragma unroll
    for (int q = 0; q < SB; ++q) {
      const int s = b * SB + q;
      if (MODE == kOrdDen)
        a.out[j] = acc[i][0];
      else if (s < a.n)
        a.out[(int64_t)s * NN + j] = acc[i][q];
    }
  }
}

template <int PW, int PH, int SB, int MODE>
hipError_t ord_launch(const OrdArgs &a, bool exact, hipStream_t st) {
  const int N = a.g.N;
  const int sxn = (N + PW - 1) / PW, syn = (N + PH - 1) / PH;
  const int blocks = ((sxn + kOrdStrips - 1) / kOrdStrips) * ((syn + kOrdStrips - 1) / kOrdStrips);
  const int nb = MODE == kOrdDen ? 1 : (a.n + SB - 1) / SB;
  if (exact)
    hipLaunchKernelGGL((k_bp_ordered<PW, PH, SB, MODE, true>), dim3(blocks, nb),
                       dim3(kOrdBlock), 0, st, a);
  else
    hipLaunchKernelGGL((k_bp_ordered<PW, PH, SB, MODE, false>), dim3(blocks, nb),
                       dim3(kOrdBlock), 0, st, a);
  return hipGetLastError();
}


// Tile form: see the header.  One wavefront per (8 x 8 tile, slice batch).
constexpr int kOT = 8;       // tile side
constexpr int kOA = 4;       // projections per round
constexpr int kORanks = 16;  // column slots per projection (>= the tile's count bound)
constexpr int kOSlots = 3;   // candidate columns per pixel and projection
constexpr int kODups = 2;    // segments per ray and pixel
constexpr int kOWave = 64;

// projection slot (0 .. kOA-1) of a lane's phase-1 pair
__device__ __forceinline__ int ai1_of(int lane) { return lane / kORanks; }

// Column slot of a column (>= -3): its remainder modulo 3.
__device__ __forceinline__ int column_slot(int c) { return (int)((unsigned)(c + 3) % kOSlots); }

// Segments per column slot of a pixel's count word (a nibble per segment:
// 0 or 1), two bits each, the slots in turn from m0 on.
__device__ __forceinline__ unsigned slot_counts(unsigned word, int m0) {
  const unsigned n = (word & 0x010101u) + ((word >> 4) & 0x010101u);  // a byte per slot
  const unsigned r = n | (n << 24);                                   // slot 3 = slot 0
  const unsigned n0 = (r >> (8 * m0)) & 3u;
  const unsigned n1 = (m0 == 2 ? n : r >> (8 * m0 + 8)) & 3u;
  const unsigned n2 = (m0 == 0 ? n >> 16 : (m0 == 1 ? n : n >> 8)) & 3u;
  return n0 | (n1 << 2) | (n2 << 4);
}

template <int SB>
struct OrdTileLds {
  static constexpr int kWPitch = SB >= 4 ? SB + 4 : SB;  // row pitch of s_w (bank spread)
};

template <int SB, int MODE, bool kExact>
__global__ void __launch_bounds__(kOWave)
k_bp_ordered_tile(OrdArgs a, unsigned *__restrict__ overflow) {
  static_assert(SB <= kWeightPad, "a slice batch of weights past the last row must be allocated");
  constexpr int WP = OrdTileLds<SB>::kWPitch;
  // segments filed, a nibble per (column slot, segment number)
  __shared__ unsigned s_cnt[kOA][kOWave];
  __shared__ float s_len[kOA][kOSlots * kODups][kOWave];
  __shared__ float s_w[MODE == kOrdDen ? 1 : kOA * kORanks * WP];
  __shared__ int s_cmin[kOA];
  const int N = a.g.N, C = a.g.C;
  const int tiles_x = (N + kOT - 1) / kOT;
  const int tile = (int)xcd_chunked(blockIdx.x, gridDim.x);
  const int tx0 = (tile % tiles_x) * kOT, ty0 = (tile / tiles_x) * kOT;
  const int tx1 = min(tx0 + kOT, N), ty1 = min(ty0 + kOT, N);
  const int b = blockIdx.y;
  const int lane = threadIdx.x;
  const int64_t NN = (int64_t)N * N;
  // the pixel this lane sums
  const int px = tx0 + (lane % kOT), py = ty0 + (lane / kOT);
  const bool pix_ok = px < N && py < N;
  const float pcx0 = grid_line(N, px), pcx1 = grid_line(N, px + 1);
  const float pcy0 = grid_line(N, py), pcy1 = grid_line(N, py + 1);
  float acc[SB], xv[SB];
#pragma unroll
  for (int q = 0; q < SB; ++q) acc[q] = 0.f, xv[q] = 0.f;
  if (MODE == kOrdNum && pix_ok) {
    const int s0 = b * SB;
    const float *src =
        a.xb + ((int64_t)(s0 / a.xsb) * NN + (int64_t)py * N + px) * a.xsb + s0 % a.xsb;
#pragma unroll
    for (int q = 0; q < SB; ++q) xv[q] = src[q];
  }
  // Wait for the pixel's values here, once.  Otherwise the compiler waits
  // for them where phase 2 first reads them, inside the loop, and its
  // in-order counter then also waits for the next round's prefetch issued
  // just before, which serialises every round on that fetch.
  wait_vector_loads();
  const float x0 = grid_line(N, tx0), x1 = grid_line(N, tx1);
  const float y0 = grid_line(N, ty0), y1 = grid_line(N, ty1);
  // The angle records of the next round are loaded at the start of a round
  // (nxt: the four projections, for the pixels' columns; fang: this lane's
  // phase-1 projection, for its pair), so that they have arrived by the
  // time they are used and their wait never covers the pair prefetch.
  AngleInfo nxt[kOA], fang;
  auto load_angles = [&](int p) {
#pragma unroll
    for (int ai = 0; ai < kOA; ++ai) nxt[ai] = a.ang[min(p + ai, a.P - 1)];
    fang = a.ang[min(p + ai1_of(lane), a.P - 1)];
  };
  // this lane's pixel's first candidate column for a round's projections, and
  // that column modulo 3 (columns are not negative where a ray exists)
  int pc0[kOA], pm0[kOA];
  auto pixel_columns = [&](int p) {
#pragma unroll
    for (int ai = 0; ai < kOA; ++ai) {
      int c0 = 0, c1;
      if (p + ai < a.P) tile_columns(nxt[ai], pcx0, pcx1, pcy0, pcy1, a.yi0, c0, c1);
      pc0[ai] = c0;
      pm0[ai] = column_slot(c0);
    }
  };
#pragma unroll
  for (int ai = 0; ai < kOA; ++ai) s_cnt[ai][lane] = 0;
  load_angles(0);
  pixel_columns(0);
  __syncthreads();
  const int ai1 = ai1_of(lane), k1 = lane % kORanks;  // phase-1 pair of this lane
  // The lane's phase-1 pair of a round, fetched one round ahead: its ray
  // table entry and weights mostly miss L2, so the next round's loads are
  // issued before this round's phase 2 and arrive while it runs.
  struct Pair {
    int c, cmin, quadrant;
    bool ok;
    RayInfo ray;
    float w[SB];
  };
  // Every lane issues the same loads on every path (row 0 when it has no
  // pair; a whole slice batch of weights, which the kWeightPad floats after
  // the weights keep in bounds for the last row): with one path, the
  // compiler's wait for a load covers that load and the older ones only, so
  // the prefetch is never waited for before its use.
  auto fetch = [&](int p, const AngleInfo &ang, Pair &q) {
    int cmin, cmax;
    tile_columns(ang, x0, x1, y0, y1, a.yi0, cmin, cmax);
    q.cmin = cmin;
    q.quadrant = ang.quadrant;
    q.c = cmin + k1;
    q.ok = p < a.P && q.c <= cmax && q.c >= 0 && q.c < C;
    const int64_t t = q.ok ? (int64_t)p * C + q.c : 0;
    q.ray = a.rays[t];
    if (MODE != kOrdDen) {
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
  Pair cur;
  fetch(ai1, fang, cur);
  for (int p0 = 0; p0 < a.P; p0 += kOA) {
    load_angles(p0 + kOA);
    // phase 1: walk the pairs, file each segment of the tile in its slot
    const int p = p0 + ai1;
    if (p < a.P) {
      if (k1 == 0) s_cmin[ai1] = cur.cmin;
      if (cur.ok) {
        const int c = cur.c;
        if (MODE != kOrdDen) {
          // slots past the stack's last slice (read from the next row) add 0
          float *dst = s_w + (ai1 * kORanks + k1) * WP;
#pragma unroll
          for (int q = 0; q < SB; ++q) dst[q] = b * SB + q < a.n ? cur.w[q] : 0.f;
        }
        const int slot = column_slot(c);
        float *len0 = &s_len[ai1][slot * kODups][0];
        const unsigned one0 = 1u << (8 * slot);
        int last = -1, again = 0;  // the pixel filed last, and its segment number
        traverse_window<kExact, true>(a.g, cur.ray, cur.quadrant, tx0, tx1, ty0, ty1,
                                      [&](int ix, int iy, float l, float) {
          const unsigned lx = (unsigned)(ix - tx0), ly = (unsigned)(iy - ty0);
          if (lx < (unsigned)(tx1 - tx0) && ly < (unsigned)(ty1 - ty0)) {
            const int lp = (int)(ly * kOT + lx);
            // a third segment (or a return to a pixel left) counts past 1 in
            // its nibble, which phase 2 reports
            again = lp == last ? 1 : 0;
            last = lp;
            len0[again * kOWave + lp] = l;
            atomicAdd(&s_cnt[ai1][lp], again ? one0 << 4 : one0);
          }
        });
      }
    }
    __syncthreads();
    fetch(p0 + kOA + ai1, fang, cur);  // next round's pair, in flight during phase 2
    // phase 2: each lane adds its pixel's segments in order, (projection,
    // column slot, segment) ascending.  With many slices per segment the
    // lane's segments of the round are walked by one flat loop, so that the
    // wavefront runs as many iterations as its busiest pixel has segments
    // rather than one per slot that any lane uses; with few slices the
    // decoding would cost more than it saves, and the loops nest.
    // `slot` counts from the pixel's first column, m0 is that one's place
    auto add = [&](int ai, int kbase, int m0, int slot, int d) {
      const int at = m0 + slot - (m0 + slot >= kOSlots ? kOSlots : 0);
      const float l = s_len[ai][at * kODups + d][lane];
      if (MODE == kOrdDen) {
        acc[0] = acc[0] + l;
      } else {
        const float *wr = s_w + (ai * kORanks + kbase + slot) * WP;
#pragma unroll
        for (int q = 0; q < SB; ++q) {
          if (MODE == kOrdEM)
            acc[q] = acc[q] + l * wr[q];
          else
            acc[q] = acc[q] - (xv[q] * l) * wr[q];
        }
      }
    };
    if (pix_ok && SB >= 8) {
      static_assert(kOSlots == 3 && kODups <= 3, "two-bit counts of three slots");
      unsigned cnt[kOA];  // n0 | n1 << 2 | n2 << 4 per projection, from its first column on
      int kb[kOA], end[kOA];
      int total = 0;
#pragma unroll
      for (int ai = 0; ai < kOA; ++ai) {
        const unsigned n = slot_counts(s_cnt[ai][lane], pm0[ai]);
        cnt[ai] = n;
        total += (int)((n & 3u) + ((n >> 2) & 3u) + (n >> 4));
        end[ai] = total;
        kb[ai] = pc0[ai] - s_cmin[ai];
      }
      for (int k = 0; k < total; ++k) {
        // projection of the k-th segment, and its rank r within it
        int ai = 0, base = 0;
#pragma unroll
        for (int i = 0; i < kOA - 1; ++i)
          if (k >= end[i]) ai = i + 1, base = end[i];
        unsigned c = cnt[0];
        int kbase = kb[0], m0 = pm0[0];
#pragma unroll
        for (int i = 1; i < kOA; ++i)
          if (ai == i) c = cnt[i], kbase = kb[i], m0 = pm0[i];
        const int r = k - base;
        const int n0 = (int)(c & 3u), n01 = n0 + (int)((c >> 2) & 3u);
        const int slot = (r >= n0) + (r >= n01);
        add(ai, kbase, m0, slot, r - (slot == 0 ? 0 : (slot == 1 ? n0 : n01)));
      }
    } else if (pix_ok) {
#pragma unroll
      for (int ai = 0; ai < kOA; ++ai) {
        const unsigned word = s_cnt[ai][lane];
        if (word == 0) continue;
        const unsigned n = slot_counts(word, pm0[ai]);
        const int kbase = pc0[ai] - s_cmin[ai];
#pragma unroll
        for (int slot = 0; slot < kOSlots; ++slot) {
          const int ns = (int)((n >> (2 * slot)) & 3u);
          for (int d = 0; d < ns; ++d) add(ai, kbase, pm0[ai], slot, d);
        }
      }
    }
#pragma unroll
    for (int ai = 0; ai < kOA; ++ai) {
      if (s_cnt[ai][lane] & 0xEEEEEEEEu) atomicOr(overflow, 1u);
      s_cnt[ai][lane] = 0;
    }
    pixel_columns(p0 + kOA);
    __syncthreads();
  }
  if (!pix_ok) return;
  const int64_t j = (int64_t)py * N + px;
  if (MODE == kOrdDen) {
    a.out[j] = acc[0];
    return;
  }
#pragma unroll
  for (int q = 0; q < SB; ++q)
    if (b * SB + q < a.n) a.out[(int64_t)(b * SB + q) * NN + j] = acc[q];
}

// LDS of W wavefronts summing SB slices.
template <int SB, int W, bool kGrid>
struct OrdSharedLds {
  static constexpr int kPitch = SB >= 4 ? SB + 4 : SB;  // row pitch of w (bank spread)
  static constexpr int kDups = kGrid ? 3 : kODups;  // segments per ray and pixel
  static constexpr int kOwn = kOA * kOSlots * kDups;
  static constexpr int kTerms = kOwn + (kGrid ? kOA * kDups : 0);  // and wrapped ones
  static constexpr int kRows = kOA * kORanks + (kGrid ? kOA : 0);
  float len[W][kTerms][kOWave];            // segment lengths in their slots
  float w[W][kRows][kPitch];               // weights of the round's rays
  unsigned cnt[W][kOA][kOWave];            // presence counts and columns (see the kernel)
  unsigned total[W][kOWave];               // segments of a pixel, per wavefront's projections
  unsigned short code[W][kTerms][kOWave];  // their places in order: len row | w row << 8
  unsigned edge[kGrid ? W : 1][kOA][kOT]; // wrapped segments of a row, and 1 << 8 if first
};

// The tile form for small images: a workgroup of W wavefronts per (tile, slice
// batch).  With one wavefront a tile, an image of few tiles spends its time in
// rounds that follow one another, four projections each, and splitting the
// batch to have more wavefronts repeats the walks.  Here each wavefront files
// the segments of its own four projections of a round and lists their places in
// order, then each sums SB / W of the slices over the 4 W projections,
// ascending.  A large image is served better by one wavefront a tile, which
// holds less LDS and waits for no other.
//
// kGrid: the geometry may have rays on grid lines.  A crossing of such a ray
// can be computed tens of pixels away, so the ray comes back to pixels it has
// left, and its segments are numbered by the count so far.  On the right edge
// line its segments wrap (ix == N) into column 0, whose tiles also take the
// flagged rays through the strip left of the edge, a column a projection at
// most, and list a wrapped segment before or after the pixel's own by its
// column.  Anything else sets the overflow flag, and the per-pixel form is used.
template <int SB, int W, int MODE, bool kExact, bool kGrid>
__global__ void __launch_bounds__(kOWave * W)
k_bp_ordered_shared(OrdArgs a, unsigned *__restrict__ overflow) {
  static_assert(SB <= kWeightPad, "a slice batch of weights past the last row must be allocated");
  constexpr int SBW = SB > W ? SB / W : 1;  // slices a wavefront sums
  using Lds = OrdSharedLds<SB, W, kGrid>;
  extern __shared__ __align__(16) unsigned char s_raw[];
  auto &lds = *reinterpret_cast<Lds *>(s_raw);
  const int N = a.g.N, C = a.g.C;
  const int tiles_x = (N + kOT - 1) / kOT;
  const int tile = (int)xcd_chunked(blockIdx.x, gridDim.x);
  const int tx0 = (tile % tiles_x) * kOT, ty0 = (tile / tiles_x) * kOT;
  const int tx1 = min(tx0 + kOT, N), ty1 = min(ty0 + kOT, N);
  const int b = blockIdx.y;
  const int lane = threadIdx.x % kOWave;
  const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kOWave);
  const int64_t NN = (int64_t)N * N;
  // the pixel this lane sums, and its first slice
  const int px = tx0 + (lane % kOT), py = ty0 + (lane / kOT);
  const bool pix_ok = px < N && py < N && wv * SBW < SB;
  const int s0 = b * SB + wv * SBW;
  const float pcx0 = grid_line(N, px), pcx1 = grid_line(N, px + 1);
  const float pcy0 = grid_line(N, py), pcy1 = grid_line(N, py + 1);
  float acc[SBW], xv[SBW];
#pragma unroll
  for (int q = 0; q < SBW; ++q) acc[q] = 0.f, xv[q] = 0.f;
  if (MODE == kOrdNum && pix_ok) {
    const float *src =
        a.xb + ((int64_t)(s0 / a.xsb) * NN + (int64_t)py * N + px) * a.xsb + s0 % a.xsb;
#pragma unroll
    for (int q = 0; q < SBW; ++q) xv[q] = src[q];
  }
  // Wait for the pixel's values here, once.  Otherwise the compiler waits
  // for them where phase 3 first reads them, inside the loop, and its
  // in-order counter then also waits for the next round's prefetch issued
  // just before, which serialises every round on that fetch.
  wait_vector_loads();
  const float x0 = grid_line(N, tx0), x1 = grid_line(N, tx1);
  const float y0 = grid_line(N, ty0), y1 = grid_line(N, ty1);
  const int ai1 = lane / kORanks, k1 = lane % kORanks;  // phase-1 pair of this lane
  // The angle records of the next round are loaded at the start of a round
  // (nxt: this wavefront's four projections, for the pixels' columns; fang:
  // this lane's phase-1 projection, for its pair), so that they have arrived
  // by the time they are used and their wait never covers the pair prefetch.
  AngleInfo nxt[kOA], fang;
  auto load_angles = [&](int p) {
#pragma unroll
    for (int ai = 0; ai < kOA; ++ai) nxt[ai] = a.ang[min(p + ai, a.P - 1)];
    fang = a.ang[min(p + ai1, a.P - 1)];
  };
  // The lane's phase-1 pair of a round, fetched one round ahead: its ray
  // table entry and weights mostly miss L2, so the next round's loads are
  // issued before this round's sums and arrive while they run.
  struct Pair {
    int c, cmin, quadrant;
    bool ok;
    RayInfo ray;
    float w[SB];
  };
  // Every lane issues the same loads on every path (row 0 when it has no
  // pair; a whole slice batch of weights, which the kWeightPad floats after
  // the weights keep in bounds for the last row): with one path, the
  // compiler's wait for a load covers that load and the older ones only, so
  // the prefetch is never waited for before its use.
  auto fetch = [&](int p, const AngleInfo &ang, Pair &q) {
    int cmin, cmax;
    tile_columns(ang, x0, x1, y0, y1, a.yi0, cmin, cmax);
    q.cmin = cmin;
    q.quadrant = ang.quadrant;
    q.c = cmin + k1;
    q.ok = p < a.P && q.c <= cmax && q.c >= 0 && q.c < C;
    const int64_t t = q.ok ? (int64_t)p * C + q.c : 0;
    q.ray = a.rays[t];
    if (MODE != kOrdDen) {
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
  Pair cur;
  // Count words of a round: in the low 24 bits a byte per column slot, with a
  // nibble per segment number (kGrid: the number of segments); above them the pixel's first candidate column counted from
  // the tile's (plus one), and that column modulo 3.
  auto start_counts = [&](int p) {
#pragma unroll
    for (int ai = 0; ai < kOA; ++ai) {
      int c0 = 0, c1;
      if (p + ai < a.P) tile_columns(nxt[ai], pcx0, pcx1, pcy0, pcy1, a.yi0, c0, c1);
      const int cmin = __builtin_amdgcn_readlane(cur.cmin, ai * kORanks);
      lds.cnt[wv][ai][lane] =
          ((unsigned)(c0 - cmin + 1) << 26) | ((unsigned)column_slot(c0) << 24);
    }
    if (kGrid && lane < kOA * kOT) lds.edge[wv][lane / kOT][lane % kOT] = 0;
  };
  // Files the wrapped segments of this wavefront's projections: lane (ai1, k1)
  // takes the k1-th column through the strip.
  auto file_wrapped = [&](int p0, int p, const AngleInfo &ang) {
    int emin, emax;
    tile_columns(ang, grid_line(N, N - 1), grid_line(N, N), grid_line(N, ty0 - 1), y1, a.yi0, emin,
                 emax);
    const int c = emin + k1;
    bool ok = p < a.P && c <= emax && c >= 0 && c < C;
    const int64_t t = ok ? (int64_t)p * C + c : 0;
    const RayInfo ray = a.rays[t];
    ok = ok && (ray.alo & kRayWraps);
    const uint64_t mine = (__ballot(ok) >> (ai1 * kORanks)) & 0xFFFFu;
    if (!ok) return;
    int cmin, cmax;
    tile_columns(ang, x0, x1, y0, y1, a.yi0, cmin, cmax);
    if (emax - emin >= kORanks || __popcll(mine) > 1 || (c >= cmin && c <= cmax)) {
      atomicOr(overflow, 1u);
      return;
    }
    if (MODE != kOrdDen) {
      const float *wr = a.w + t * a.S + b * SB;
      float *dst = lds.w[wv][kOA * kORanks + ai1];
      for (int q = 0; q < SB; ++q) dst[q] = b * SB + q < a.n ? wr[q] : 0.f;
    }
    traverse_window<kExact, true>(a.g, ray, ang.quadrant, N - 1, N, ty0 - 1, ty1,
                                  [&](int ix, int iy, float l, float) {
      const unsigned ly = (unsigned)(iy + 1 - ty0);
      if (ix == N && ly < (unsigned)(ty1 - ty0)) {
        unsigned &n = lds.edge[wv][ai1][ly];
        const unsigned k = n & 0xFFu;
        if (k < Lds::kDups) lds.len[wv][Lds::kOwn + ai1 * Lds::kDups + k][ly * kOT] = l;
        n = (n + 1) | (c < cmin ? 0x100u : 0u);
      }
    });
  };
  constexpr int kRound = kOA * W;  // projections per round
  AngleInfo fcur;  // this round's fang
  load_angles(wv * kOA);
  fcur = fang;
  fetch(wv * kOA + ai1, fang, cur);
  start_counts(wv * kOA);
  for (int r0 = 0; r0 < a.P; r0 += kRound) {
    const int p0 = r0 + wv * kOA;  // this wavefront's first projection
    if (kGrid) fcur = fang;
    load_angles(p0 + kRound);
    // phase 1: walk the pairs, file each segment of the tile in its slot
    const int p = p0 + ai1;
    if (p < a.P && cur.ok) {
      const int c = cur.c;
      if (MODE != kOrdDen) {
        // slots past the stack's last slice (read from the next row) add 0
        float *dst = lds.w[wv][lane];
#pragma unroll
        for (int q = 0; q < SB; ++q) dst[q] = b * SB + q < a.n ? cur.w[q] : 0.f;
      }
      const int slot = column_slot(c);
      float *len0 = lds.len[wv][(ai1 * kOSlots + slot) * Lds::kDups];
      const unsigned one0 = 1u << (8 * slot);
      int last = -1, again = 0;  // the pixel filed last, and its segment number
      traverse_window<kExact, true>(a.g, cur.ray, cur.quadrant, tx0, tx1, ty0, ty1,
                                    [&](int ix, int iy, float l, float) {
        const unsigned lx = (unsigned)(ix - tx0), ly = (unsigned)(iy - ty0);
        if (lx < (unsigned)(tx1 - tx0) && ly < (unsigned)(ty1 - ty0)) {
          const int lp = (int)(ly * kOT + lx);
          unsigned *cnt = &lds.cnt[wv][ai1][lp];
          if constexpr (kGrid) {
            // only this lane counts in its slot's byte
            const int k = (int)((*cnt >> (8 * slot)) & 0xFFu);
            if (k < Lds::kDups) len0[k * kOWave + lp] = l;
            if (k <= Lds::kDups) atomicAdd(cnt, one0);
          } else {
            // a third segment (or a return to a pixel left) counts past 1 in
            // its nibble, which phase 2 reports
            again = lp == last ? 1 : 0;
            last = lp;
            len0[again * kOWave + lp] = l;
            atomicAdd(cnt, again ? one0 << 4 : one0);
          }
        }
      });
    }
    if (kGrid && tx0 == 0) file_wrapped(p0, p, fcur);
    // Phase 2: each lane lists the places of its pixel's segments of this
    // wavefront's projections in order, (projection, column, segment)
    // ascending.  Only this wavefront has filed there, and its LDS accesses
    // take effect in the order they are issued.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    {
      unsigned short *dst = &lds.code[wv][0][lane];
      int n = 0;
#pragma unroll
      for (int ai = 0; ai < kOA; ++ai) {
        const unsigned word = lds.cnt[wv][ai][lane];
        if (!kGrid && (word & 0x00EEEEEEu)) atomicOr(overflow, 1u);
        unsigned wrapped = 0;
        if (kGrid && lane % kOT == 0) wrapped = lds.edge[wv][ai][lane / kOT];
        if ((wrapped & 0xFFu) > Lds::kDups) atomicOr(overflow, 1u);
        auto list_wrapped = [&]() {
          for (unsigned k = 0; k < (wrapped & 0xFFu) && k < Lds::kDups; ++k) {
            *dst = (unsigned short)((Lds::kOwn + ai * Lds::kDups + k) |
                                    ((kOA * kORanks + ai) << 8));
            dst += kOWave, ++n;
          }
        };
        if (kGrid && (wrapped & 0x100u)) list_wrapped();
        unsigned at = (word >> 24) & 3u;            // slot of the candidate column
        unsigned row = ai * kORanks + (word >> 26) - 1;  // and its pair
#pragma unroll
        for (int k = 0; k < kOSlots; ++k) {
          const unsigned has = word >> (8 * at);
          const unsigned code = (ai * kOSlots + at) * Lds::kDups | (row << 8);
          if constexpr (kGrid) {
            const unsigned m = has & 0xFFu;
            if (m > Lds::kDups) atomicOr(overflow, 1u);
            for (unsigned d = 0; d < m && d < Lds::kDups; ++d) {
              *dst = (unsigned short)(code + d);
              dst += kOWave, ++n;
            }
          } else {
            if (has & 0x01u) {
              *dst = (unsigned short)code;
              dst += kOWave, ++n;
            }
            if (has & 0x10u) {
              *dst = (unsigned short)(code + 1);
              dst += kOWave, ++n;
            }
          }
          at = at == kOSlots - 1 ? 0 : at + 1;
          ++row;
        }
        if (kGrid && wrapped && !(wrapped & 0x100u)) list_wrapped();
      }
      lds.total[wv][lane] = n;
    }
    __syncthreads();
    fetch(p0 + kRound + ai1, fang, cur);  // next round's pair, in flight during phase 3
    // phase 3: each lane adds its pixel's segments, the wavefronts' projections
    // in turn; as many iterations as the busiest pixel has segments
    if (pix_ok) {
      for (int g = 0; g < W; ++g) {
        const int n = (int)lds.total[g][lane];
        const unsigned short *src = &lds.code[g][0][lane];
        const float *len = &lds.len[g][0][lane];
        const float *wg = &lds.w[g][0][MODE == kOrdDen ? 0 : wv * SBW];
        for (int k = 0; k < n; ++k) {
          const unsigned code = *src;
          src += kOWave;
          const float l = len[(code & 0xFFu) * kOWave];
          if (MODE == kOrdDen) {
            acc[0] = acc[0] + l;
          } else {
            const float *wr = wg + (code >> 8) * Lds::kPitch;
#pragma unroll
            for (int q = 0; q < SBW; ++q) {
              if (MODE == kOrdEM)
                acc[q] = acc[q] + l * wr[q];
              else
                acc[q] = acc[q] - (xv[q] * l) * wr[q];
            }
          }
        }
      }
    }
    __syncthreads();
    start_counts(p0 + kRound);
  }
  if (!pix_ok) return;
  const int64_t j = (int64_t)py * N + px;
  if (MODE == kOrdDen) {
    a.out[j] = acc[0];
    return;
  }
#pragma unroll
  for (int q = 0; q < SBW; ++q)
    if (s0 + q < a.n) a.out[(int64_t)(s0 + q) * NN + j] = acc[q];
}

template <int SB, int W, int MODE, bool kGrid>
hipError_t ord_shared_launch(const OrdArgs &a, bool exact, unsigned *overflow, hipStream_t st) {
  const int N = a.g.N;
  const int tiles = ((N + kOT - 1) / kOT) * ((N + kOT - 1) / kOT);
  const int nb = MODE == kOrdDen ? 1 : (a.n + SB - 1) / SB;
  constexpr size_t lds = sizeof(OrdSharedLds<SB, W, kGrid>);
  static_assert(lds <= 160 * 1024, "a workgroup's LDS");
  auto kern = exact ? k_bp_ordered_shared<SB, W, MODE, true, kGrid>
                    : k_bp_ordered_shared<SB, W, MODE, false, kGrid>;
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute(
        (const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kern, dim3(tiles, nb), dim3(kOWave * W), lds, st, a, overflow);
  return hipGetLastError();
}

template <int SB, int MODE>
hipError_t ord_tile_launch(const OrdArgs &a, bool exact, unsigned *overflow, hipStream_t st) {
  const int N = a.g.N;
  const int tiles = ((N + kOT - 1) / kOT) * ((N + kOT - 1) / kOT);
  const int nb = MODE == kOrdDen ? 1 : (a.n + SB - 1) / SB;
  if (exact)
    hipLaunchKernelGGL((k_bp_ordered_tile<SB, MODE, true>), dim3(tiles, nb), dim3(kOWave), 0, st,
                       a, overflow);
  else
    hipLaunchKernelGGL((k_bp_ordered_tile<SB, MODE, false>), dim3(tiles, nb), dim3(kOWave), 0,
                       st, a, overflow);
  return hipGetLastError();
}

}  // namespace

// Wavefronts per tile: more where the tiles alone leave the GPU's SIMDs idle.
// One launch with 1 / 4 / 8, PML num (us):
//    59^2,  700 angles   1 slice 967 / 344 /  237   32 slices 1344 /  445 /  340
//   151^2,  400                  590 / 213 /  269              792 /  279 /  377
//   300^2,  300                  471 / 345 /  589              686 /  610 /  802
//   400^2,  300                  547 / 622 /  997             1220 / 1005 / 1358
//   511^2,  200                  498 / 639 / 1110              916 / 1102 / 1487
// Tiles of geometries with rays on grid lines always share (129^2, 110 angles, 11
// slices: 175 us, 745 in the per-pixel form; den of 125^2, 122 angles 94, per pixel
// 2131).
int ordered_waves(int N, int S, int sb, bool grid_rays) {
  const int64_t tiles =
      (int64_t)((N + kOT - 1) / kOT) * ((N + kOT - 1) / kOT) * ((S + sb - 1) / sb);
  if (grid_rays) return 4;
  return tiles <= 128 ? 8 : (tiles <= (sb == 32 ? 3000 : 1536) ? 4 : 1);
}

// Whether rays on grid lines are served faster by the tile form than pixel by
// pixel.  Such a ray is walked whole in every tile it touches, which costs N^2 a
// ray (a tenth to a quarter of it in the per-pixel form, whose threads walk it side
// by side), and so do rays whose lists are not sorted; an angle costs N^2 in tiles,
// and in the per-pixel form N^2 or, where its strips do not fill the GPU, the walks
// of one (`least`).  Costs in us of a batch: sb slices in tiles, up to 8 per pixel,
// fitted to ten sides at 120, 360 and 900 angles: where the two forms differ by
// more than 5% the faster is chosen in all but one of 196 cases (the costs are
// within 4 and 16% of the measured times on average).  Tile /
// per-pixel form (ms), one angle's rays on grid lines, angles 120, 360, 900:
//              column sums                    num of 1 or 2 slices
//    512^2   1.1 / 2.3  2.2 / 6.4  4.5 / 15   1.1 / 1.6  2.2 / 4.2  4.7 / 10
//    640^2   1.9 / 1.5  3.5 / 4.0  7.3 / 9.5  1.9 / 1.8  3.6 / 4.7  7.5 / 11
//    900^2   4.4 / 2.7  7.7 / 6.8   15 / 16   4.5 / 3.3  7.8 / 8.4   15 / 19
//   1200^2   9.2 / 3.0   15 / 7.3   28 / 17   9.3 / 5.6   15 / 13    28 / 31
//   2048^2    39 / 9.8   55 / 19              39 / 20     56 / 42
//              num of 4 or 8                  num of 32
//    384^2   1.1 / 1.5  2.2 / 4.1  4.9 / 10   1.2 / 3.2  2.7 / 9.6  6.0 / 23
//    512^2   2.1 / 1.7  4.2 / 4.4  8.9 / 11   2.4 / 5.1  5.0 / 15    11 / 36
//    640^2   3.5 / 1.8  6.8 / 4.7   14 / 11   4.1 / 6.5  8.2 / 19    17 / 47
//   2048^2    73 / 19   106 / 42              81 / 80    122 / 190
// A launch also holds fewer than 2^32 lanes, which four wavefronts a tile reach
// at 32761^2.
bool ordered_grid_pays(int N, int P, int64_t whole, int S, int mode, int sb) {
  const int64_t side = (N + kOT - 1) / kOT;
  if (side * side * kOWave * ordered_waves(N, 1, 1, true) >= (int64_t(1) << 32)) return false;
  struct Cost {
    double tile_ray, tile, pixel_ray, pixel, least;
  };
  const Cost c = mode == kOrdDen ? Cost{3.7e-6, 1.63e-5, 0.57e-6, 0.98e-5, 17.5}
                 : sb <= 2       ? Cost{3.7e-6, 1.72e-5, 1.0e-6, 2.45e-5, 9}
                 : sb <= 8       ? Cost{6.7e-6, 3.3e-5, 0.95e-6, 2.4e-5, 11.5}
                 : sb == 16      ? Cost{7.0e-6, 3.46e-5, 0.9e-6, 2.5e-5, 9.3}
                                 : Cost{7.03e-6, 4.09e-5, 0.71e-6, 2.74e-5, 10};
  const double n2 = (double)N * N, rays = n2 * (double)whole;
  const int tiles = mode == kOrdDen ? 1 : (S + sb - 1) / sb, pixels = mode == kOrdDen ? 1 : (S + 7) / 8;
  return tiles * (c.tile_ray * rays + c.tile * n2 * P) <=
         pixels * (c.pixel_ray * rays + std::fmax(c.least, c.pixel * n2) * P);
}

bool ordered_sb_supported(int mode, int sb, int xsb) {
  if (mode == kOrdDen) return true;
  if (sb != 1 && sb != 2 && sb != 4 && sb != 8 && sb != 16 && sb != 32) return false;
  return mode == kOrdEM || (xsb >= sb && xsb % sb == 0);
}

hipError_t launch_bp_ordered(const Geometry &g, const RayInfo *rays, int mode, bool exact,
                             const float *w, const float *xb, int xsb, int sb, float *out,
                             bool wraps, unsigned *tile_overflow, bool grid_rays,
                             int s0, int n, hipStream_t st) {
  OrdArgs a;
  a.g = g.grid;
  a.ang = g.d_ang;
  a.rays = rays;
  a.P = g.P;
  a.S = g.S;
  a.n = n;
  a.yi0 = g.yi0;
  a.w = w ? w + s0 : nullptr;
  // a slot batch of the copy, and the slots within it (the kernels step from
  // there by sb, which divides xsb)
  a.xb = xb ? xb + (int64_t)(s0 / xsb) * g.NN() * xsb + s0 % xsb : nullptr;
  a.xsb = xsb;
  a.out = out + (int64_t)s0 * g.NN();
  a.wraps = wraps ? 1 : 0;
  if (!ordered_sb_supported(mode, sb, xsb)) return hipErrorInvalidValue;
  if (tile_overflow) {
    // tile form; wrapped segments need the grid-ray one
    if (wraps && !grid_rays) return hipErrorInvalidValue;
    const int waves = ordered_waves(g.N, mode == kOrdDen ? 1 : n, sb, grid_rays);
#define TRACE_ORDS_CASE(SB_, W_, GRID_)                                                     \
  if (waves == W_ && grid_rays == GRID_) {                                                      \
    if (mode == kOrdDen)                                                                     \
      return ord_shared_launch<1, W_, kOrdDen, GRID_>(a, exact, tile_overflow, st);         \
    if (sb == SB_)                                                                           \
      return mode == kOrdNum                                                                 \
                 ? ord_shared_launch<SB_, W_, kOrdNum, GRID_>(a, exact, tile_overflow, st)  \
                 : ord_shared_launch<SB_, W_, kOrdEM, GRID_>(a, exact, tile_overflow, st);  \
  }
#define TRACE_ORDS_WAVES(W_, GRID_)                                                         \
  TRACE_ORDS_CASE(1, W_, GRID_) TRACE_ORDS_CASE(2, W_, GRID_) TRACE_ORDS_CASE(4, W_, GRID_) \
  TRACE_ORDS_CASE(8, W_, GRID_) TRACE_ORDS_CASE(16, W_, GRID_) TRACE_ORDS_CASE(32, W_, GRID_)
    TRACE_ORDS_WAVES(4, false)
    TRACE_ORDS_WAVES(8, false)
    TRACE_ORDS_WAVES(4, true)
#undef TRACE_ORDS_WAVES
#undef TRACE_ORDS_CASE
    if (grid_rays) return hipErrorInvalidValue;
    if (mode == kOrdDen) return ord_tile_launch<1, kOrdDen>(a, exact, tile_overflow, st);
#define TRACE_ORDT_CASE(SB_)                                                               \
  case SB_:                                                                                \
    return mode == kOrdNum ? ord_tile_launch<SB_, kOrdNum>(a, exact, tile_overflow, st)    \
                           : ord_tile_launch<SB_, kOrdEM>(a, exact, tile_overflow, st);
    switch (sb) {
      TRACE_ORDT_CASE(1)
      TRACE_ORDT_CASE(2)
      TRACE_ORDT_CASE(4)
      TRACE_ORDT_CASE(8)
      TRACE_ORDT_CASE(16)
      TRACE_ORDT_CASE(32)
      default: return hipErrorInvalidValue;
    }
#undef TRACE_ORDT_CASE
  }
  if (sb > 8) return hipErrorInvalidValue;
  if (mode == kOrdDen) return ord_launch<2, 2, 1, kOrdDen>(a, exact, st);
#define TRACE_ORD_CASE(SB_)                                                              \
  case SB_:                                                                              \
    return mode == kOrdNum ? ord_launch<1, 1, SB_, kOrdNum>(a, exact, st)                \
                           : ord_launch<1, 1, SB_, kOrdEM>(a, exact, st);
  switch (sb) {
    TRACE_ORD_CASE(1)
    TRACE_ORD_CASE(2)
    TRACE_ORD_CASE(4)
    TRACE_ORD_CASE(8)
    default: return hipErrorInvalidValue;
  }
#undef TRACE_ORD_CASE
}

}  // namespace trace_hip
