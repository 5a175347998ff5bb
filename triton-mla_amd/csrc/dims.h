// The matrix-core decode of other head dims and of float32
// (mla_decode_dims.hip), as mla_decode_generic.hip calls it.
#pragma once

#include <hip/hip_runtime.h>

#include "decode_common.h"

namespace tmla {
namespace dims {

// PartialArgs with the capacity the lengths are cut to and the float32
// partials: [slots, heads, dv] rows and [slots, heads] base-2 log-sum-exps
// (mid_o / mid_lse are not used).
struct DimsArgs : PartialArgs {
  int32_t len_cap;
  int32_t uni;  // 1: 32 aligned tokens (float32: 16) lie in one page, less than 2^31 bytes from first to last
  float* part;
  float* part_lse;
};

// Both stages on `st`; dims accepted by dims_form (host_plan.h).
hipError_t launch(const DimsArgs& a, int dv, int dr, int dtype, int64_t capacity_tokens, hipStream_t st);

}  // namespace dims
}  // namespace tmla
