// The mid-size fp8 expert GEMMs (gemm_fp8_mid.hip) and the entry points that run them
// (gemm_fp8.hip on row tiles, the layer on block tiles).
#pragma once

#include "moe_common.h"
#include "moe_internal.h"

namespace moe {

struct MidArgs {
  const uint8_t* a;   // x codes [T, H] or h codes [rows, I]
  const float* as;    // their 1x128 scales
  const uint8_t* w;
  const float* ws;
  const uint8_t* wsh;
  const float* wssh;
  const int32_t* tpid;
  const int4* tiles;  // {expert, first slot, rows, first hq / y row}
  const int2* seg;    // block tiles: {first tile of the expert, tiles of the expert}; null: row tiles
  const int32_t* num_tiles;
  uint8_t* hq;
  float* hs;
  uint16_t* y;
  const float* cs;    // optional per-output-channel weight scales (row tiles; routed, shared)
  const float* cssh;
  int T, H, I, E, nsh;
  long NB;
  long rows;  // rows of h
};

// Whether the sizes and operands suit the kernels (kind 0 gate_up, 1 down): H and I multiples
// of 512 (whole groups of four K blocks, whole column tiles) up to 16384, aligned operands,
// and operands that 32-bit byte offsets reach. Otherwise the other kernels run.
bool mid_fits(int kind, const MidArgs& a);
// Launch on a.tiles: block tiles of at most kMidTallRows rows (a.seg set, XCD ranges in the header
// num_tiles) or row tiles of at most kMidTileRows.
void launch_mid(int kind, const MidArgs& a, int max_tiles, hipStream_t st);

}  // namespace moe
