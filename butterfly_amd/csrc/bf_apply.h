/*
 * Device-side pieces shared by the apply kernels (bf_kernels.hip,
 * bf_apply_few.hip).
 */
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bf_plan.h"

/* the vector buffers of an apply, indexed by BFK_BUF_* */
struct BfkBufs {
  const double2 *in[4];
  double2 *out[4];
};

struct BfkBufsF {
  const float2 *in[4];
  float2 *out[4];
};

template <typename V> struct BufsOf;
template <> struct BufsOf<double2> { typedef BfkBufs T; };
template <> struct BufsOf<float2> { typedef BfkBufsF T; };

/* one stage for any number of right-hand sides on the vector units
 * (bf_apply_few.hip); waves = segments per block where no segment is split
 * over waves, 0 for the default */
hipError_t bfk_launch_few(hipStream_t st, const BfkSeg *segs, int64_t numSegs, const BfkStageShape &shape,
                          const BfkTerm *terms, const double2 *arena, const BfkBufs &b, int nrhs, int waves);
hipError_t bfk_launch_few_f32(hipStream_t st, const BfkSeg *segs, int64_t numSegs, const BfkStageShape &shape,
                              const BfkTerm *terms, const float2 *hi, const float2 *lo, const BfkBufsF &b, int nrhs,
                              int waves, int sum64);
