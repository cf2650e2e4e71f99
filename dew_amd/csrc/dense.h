// What the two launches of plain bf16 operands share (bf16.hip: tiles of 64 and 128 rows; wide.hip: 256 x 256 ones).
#pragma once

#include "common.h"
#include "wide.h"

namespace dew {

struct DenseParams {
  const bf16_t* a;  // [rows, inner] (gathered), or, contracted over groups of rows, [rows, outer_m]
  const bf16_t* b;  // [groups, inner, outer_n], or [groups, outer_n, inner], or [rows, outer_n]
  const int32_t *gather, *scatter;
  const int32_t *offsets, *sizes;  // the groups of rows: their exclusive prefix [groups + 1], or their sizes
  void* out;
  const float *factor0, *factor1;  // a kernel gradient's sums times *factor0 * *factor1 (each may be null)
  int groups, rows, inner, outer_m, outer_n, m_tiles, group_m;
  int quarter_turns;  // 256 x 256 tiles: the last round in quarters where a block has at most so many
};

// 256 x 256 tiles on blocks that stay (wide.hip), of rows that are neither gathered nor scattered; `across`: a kernel gradient; `kmajor`:
// w [groups, width, depth].
int launch_wide(const char* who, const DenseParams& p, bool across, bool kmajor, bool out_f32, hipStream_t stream);

}  // namespace dew
