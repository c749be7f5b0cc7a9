// Shared by the MX expert GEMM kernels (gemm_mx.hip, gemm_mx_block.hip): the kernel
// arguments, the scaled MFMA and the activation.
#pragma once

#include <type_traits>

#include "moe_common.h"
#include "moe_internal.h"

namespace moe {

constexpr int kFmtFp8 = 0;  // MFMA format codes (cbsz / blgp) of the scaled instruction
constexpr int kFmtFp4 = 4;

struct MxArgs {
  const uint8_t* a;    // fp8 activations: x [T, H] (gate_up) or h [rows, I] (down)
  const uint8_t* as;   // their E8M0 scales [rows, K/32]
  const uint8_t* w;    // routed weights, packed (fp4: K/2 bytes per row; fp8: K)
  const uint8_t* ws;   // routed weight scales [E, rows_w, K/32]
  const float* bias;   // routed bias [E, rows_w] (fp32) or null
  const uint8_t* wsh;  // shared-expert weights / scales / bias
  const uint8_t* wssh;
  const float* bsh;
  const int32_t* tpid;
  const int4* tiles;  // {expert, first slot, rows, first hq / y row}
  const int32_t* num_tiles;
  uint8_t* hq;
  uint8_t* hs;
  uint16_t* y;
  int T, H, I, E, nsh;
  long NB;
  int act;  // 0 SiLU, 1 Swish (g * sigmoid(1.702 g))
  float gate_lo, gate_hi, up_lo, up_hi;
  // the layer at one token (tiles from its own mapping: one row each, token 0)
  int one;
  // block kernels: rows of h, and {first tile of the expert, tiles of the expert} of block
  // tiles (null: row tiles)
  long rows;
  const int2* seg;
};

// Launch of the MXFP4 block kernels (gemm_mx_block.hip; kind 0 gate_up, 1 down) on a.tiles:
// block tiles (a.seg set, XCD ranges in the header num_tiles) or row tiles, of at most
// kMxBlockTileRows rows. mx_block_fits: the sizes and operands suit them (H and I multiples
// of 512, no shared experts, 16-byte aligned operands that 32-bit byte offsets reach).
bool mx_block_fits(int kind, const MxArgs& a);
void launch_mx_block(int kind, const MxArgs& a, int max_tiles, hipStream_t st);
// Whether the MXFP4 product `kind` runs the block kernels on a list of max_tiles row tiles of mt
// rows, where mx_block_fits; otherwise the ring kernels. They run from two items per CU on, but for
// 32-row tiles of long K where three whole rounds of the ring's one workgroup per CU hold one tile
// per expert: there the block kernels' two workgroups per CU are one and a half rounds. Alone, us,
// ring -> block, 8 rows per expert: gate_up K = 3072, 512 / 640 / 704 / 768 / 800 items 44.2 / 62.5 /
// 63.5 / 64.5 / 80.9 -> 37.1 / 58.9 / 61.7 / 64.1 / 64.9; down K = 3072, 512 / 576 / 640 / 768 / 800
// items 43.4 / 57.4 / 58.3 / 61.0 / 75.8 -> 38.0 / 56.8 / 59.8 / 64.9 / 66.1; K = 1024, 768 items 27.6
// -> 23.9 and 22.8 -> 22.8. gate_up loses in whole layers (32 experts of K = 3072, 24 of K = 4096).
inline bool mx_rows_on_block(int kind, int H, int I, int E, int max_tiles, int mt) {
  const long cols = (kind == 0) ? I / 128 : H / 256;
  if ((mt != 32 && mt != 64) || max_tiles * cols < kMidMinItems) return false;
  const bool one_each = 5L * max_tiles <= 8L * E;  // up to 19 of 32 rows on average
  return !(mt == 32 && (kind == 0 ? H : I) > 2048 && one_each && E * cols > (kind == 0 ? 704 : 576) &&
           E * cols <= 768);
}

__device__ __forceinline__ v4f mfma_mx(const v8i& a, const v8i& b, const v4f& c, int sa, int sb,
                                      std::integral_constant<int, kFmtFp8>) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, kFmtFp8, kFmtFp8, 0, sa, 0, sb);
}
__device__ __forceinline__ v4f mfma_mx(const v8i& a, const v8i& b, const v4f& c, int sa, int sb,
                                      std::integral_constant<int, kFmtFp4>) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, kFmtFp8, kFmtFp4, 0, sa, 0, sb);
}

__device__ __forceinline__ float mx_act(float g, int act) {
  // hardware reciprocal (about 1 ulp): h only feeds the MXFP8 quantization
  const float k = act ? -1.702f : -1.0f;
  return g * __builtin_amdgcn_rcpf(1.0f + __expf(k * g));
}

}  // namespace moe
