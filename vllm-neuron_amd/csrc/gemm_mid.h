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

// The operands that the ring and block kernels' arguments name alike.
template <class A>
MidArgs mid_args(const A& a) {
  MidArgs m{};
  m.a = a.a;
  m.as = a.as;
  m.w = a.w;
  m.ws = a.ws;
  m.wsh = a.wsh;
  m.wssh = a.wssh;
  m.tpid = a.tpid;
  m.tiles = a.tiles;
  m.num_tiles = a.num_tiles;
  m.hq = a.hq;
  m.hs = a.hs;
  m.y = a.y;
  m.T = a.T;
  m.H = a.H;
  m.I = a.I;
  m.E = a.E;
  m.nsh = a.nsh;
  m.NB = a.NB;
  m.rows = a.NB + (long)a.nsh * a.T;
  return m;
}

// Whether the sizes and operands suit the kernels (kind 0 gate_up, 1 down): H and I multiples
// of 512 (whole groups of four K blocks, whole column tiles) up to 16384, aligned operands,
// and operands that 32-bit byte offsets reach. Otherwise the other kernels run.
bool mid_fits(int kind, const MidArgs& a);
// Whether the product `kind` runs these kernels on a list of max_tiles row tiles of mt rows, where
// mid_fits; otherwise the ring kernels. Tiles of 64 rows always: whole layer, ring -> mid-size
// kernels, DeepSeek-V3 at 257 / 600 / 1000 tokens 1850 / 2050 / 2290 -> 1769 / 1841 / 1955 us, GLM-4.5
// at 100 / 500 tokens 667 / 893 -> 610 / 681 us, Kimi-K2 at 600 / 1200 tokens 2857 / 3340 -> 2660 /
// 2841 us, the small layer at 100 tokens 49 -> 41 us. 16- and 32-row tiles only where the items fill
// the chip twice, or four times at 16 rows (GLM-4.5 30 tokens 503 -> 481 us, DeepSeek-V3 16 tokens
// 723 -> 688 us, 64 tokens 1472 -> 1427 us): below that an item is a chain of K steps, which the
// ring's three stages shorten (DeepSeek-V3 2 tokens, 272 items: 133 against 158 us; the small
// layer's 32 items at 64 tokens: 36.6 against 37.5 us; with the ring from 512 to 1024 items,
// DeepSeek-V3 at 4 / 5 / 7 tokens 292 / 314 / 395 -> 282 / 305 / 391 us and Kimi-K2 at 5 / 6 323 /
// 347 -> 317 / 343, though Kimi-K2 at 4 goes 255 -> 256 and GLM-4.5 at 5 180 -> 185). Long chains
// (gate_up of K = 7168, items counted for distinct experts) only at eight times: at 8 to 14 tokens
// (1104 to 2048 items) even routing gives the same, but with Zipf(1.2) routing the ring leads (Kimi-K2
// at 8 / 9 / 12 tokens 290 / 286 / 306 against 299 / 294 / 314 us, DeepSeek-V3 at 8 283 against 292),
// where K = 5120 gains (GLM-4.5 at 10 tokens 156 -> 146 us).
inline bool mid_rows(int kind, int H, int I, int max_tiles, int mt) {
  const long items = (long)max_tiles * (kind == 0 ? I / 128 : H / 256);
  if (mt <= 16) return items >= ((kind == 0 ? H : I) > 5120 ? 2 * kMidMinItems16 : kMidMinItems16);
  return mt == 64 || (mt == 32 && items >= kMidMinItems);
}
// Launch on a.tiles: block tiles of at most kMidTallRows rows (a.seg set, XCD ranges in the header
// num_tiles) or row tiles of at most kMidTileRows.
void launch_mid(int kind, const MidArgs& a, int max_tiles, hipStream_t st);

}  // namespace moe
