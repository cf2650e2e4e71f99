// The 256 x 256 launch of quantized rows (wide_fp8.hip).
#pragma once

#include "wide.h"

namespace dew {

struct WideFp8Params {
  const uint8_t *a, *a_scale;  // codes [rows, depth] in the instruction's operand order and scales, a_scale_pitch bytes a row; or, a kernel
                               // gradient's, a prepared bank `rows` wide
  const uint8_t* b;            // a prepared bank's codes, and its scales
  const void* b_scale;
  const int32_t* offsets;      // [groups + 1] of the rows, or (a kernel gradient) of the depth
  void* out;
  int groups, rows, depth, width, a_scale_pitch;  // a kernel gradient's `rows`: every group's
  int quarter_turns;           // the last round in quarters where a block has at most so many
};

int launch_wide_fp8(const char* who, const WideFp8Params& p, bool mx, bool gradient, bool out_f32, hipStream_t stream);

}  // namespace dew
