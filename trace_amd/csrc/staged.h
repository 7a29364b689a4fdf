// staged.h -- the slab-staged forward projector (staged.hip): host-side
// declarations.  Not part of the public interface.
#pragma once
#include <vector>

#include "internal.h"

namespace trace_hip {

// Slab-staged forward projector (staged.hip): a workgroup holds up to kStG
// angles of similar direction x kStW adjacent columns, one lane per ray, and
// sweeps the image in slabs of a few pixels, staging a window of pixels
// across each slab in LDS.
constexpr int kStG = 16;
constexpr int kStW = 64;
enum StagedAxis { kStAxisX = 0, kStAxisYUp = 1, kStAxisYDown = 2 };

// Slice batches the staged form is compiled for, and the pixels one of its
// two LDS buffers holds for each: a slab of H pixels takes a window of
// staged_pixels(sb) / H across it.  A pixel takes sb + 4 floats of LDS.
constexpr bool staged_batch(int sb) { return sb == 32 || sb == 16 || sb == 8 || sb == 4; }
constexpr int staged_pixels(int sb) {
  return sb == 32 ? 512 : (sb == 16 ? 960 : (sb == 8 ? 768 : 2048));
}

// Per-geometry plan: angle groups, and per (bundle, slab) the first pixel
// across the slab and the window's extent (0: empty).
struct StagedPlan {
  int sb = 0;             // slice batch the plan is for
  int H = 0;              // slab thickness in pixels
  int ngroups = 0, nslab = 0, ngc = 0;
  int *order = nullptr;   // [P] projections by direction
  int4 *group = nullptr;  // [ngroups] first entry of order, count, sweep axis
  int2 *range = nullptr;  // [ngroups * ngc][nslab]
};

// Angle groups and slab thickness of a geometry at slice batch sb.
struct StagedLayout {
  int H = 0;
  std::vector<int> order;
  std::vector<int4> group;
};
StagedLayout staged_layout(const Geometry &g, const AngleInfo *ang, int sb);
// Whether the staged form is the fastest one for a geometry at slice batch sb;
// `scattered`: successive projections point anywhere (scattered_angles).
bool staged_faster(const Geometry &g, int sb, bool scattered);
bool scattered_angles(const AngleInfo *ang, int P);

hipError_t launch_staged_plan(const Geometry &g, const RayInfo *rays, StagedPlan &pl,
                              hipStream_t st);
hipError_t launch_forward_staged(const Geometry &g, const RayInfo *rays, const StagedPlan &pl,
                                 int mode, bool exact, const float *xb, const float *sino,
                                 float *out, unsigned *maxw, hipStream_t st);

}  // namespace trace_hip
