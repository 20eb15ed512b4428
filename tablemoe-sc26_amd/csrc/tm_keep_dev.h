// The decoding of packed top-1 search keys into distances, shared by the
// keep selection and the search kernel that decodes its own keys.
#pragma once

#include "tm_common.h"

// Optional source of the scores: packed top-1 search keys of the layer call
// (see tm_key_to_dist) with the query norms as `parts` partial sums; the
// kernel then also writes each token's distance, centroid and |q|^2.
struct KeySrc {
  const uint64_t *keys;  // null: scores come from `score`
  const float *qn_part;  // [parts][n]
  int parts;
  int l2;
  float *out_dist;
  int64_t *out_idx;
  float *out_qn;
};

// |q|^2 from the column-group partials in the order of a lane-pair tree over
// the groups (the order a whole-row reduction across lanes adds them).
__device__ __forceinline__ float qn_sum(float a0, float a1, float a2, float a3, int parts) {
  if (parts == 1) return a0;
  if (parts == 2) return a0 + a1;
  return (a0 + a1) + (a2 + a3);
}
