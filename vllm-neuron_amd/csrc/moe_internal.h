// Host-side plumbing shared by the C-ABI entry points: error strings, argument
// checks and launch-shape helpers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <algorithm>

#include "moe_fp8.h"

namespace moe {

void set_error(const char* fn, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
void clear_error();

// K splits for the router logits GEMM: aim for >= 1024 workgroups (4 per CU
// fit, and the loop is latency-bound), each split at least 256 columns of H.
inline int router_logits_splits(int T, int H, int E) {
  long base = (long)((T + 63) / 64) * ((E + 63) / 64);
  long ks = (1024 + base - 1) / base;
  long kmax = std::max(1, H / 256);
  return (int)std::max(1L, std::min(ks, kmax));
}


// Rows per tile of the 256x256 expert GEMM kernels.
constexpr int kBlockTileRows = 256;
// Rows per tile of the prefill-sized MXFP4 expert GEMM kernels.
constexpr int kMxBlockTileRows = 128;

// Rows per tile of the mid-size fp8 expert GEMM kernels (gemm_fp8_mid.hip): row tiles, and the
// block tiles on which the layer runs them instead of the block kernels from 32 to
// kMidTallMaxRows routed rows per expert on average.
// Layer, block -> mid-size kernels, us: at 34 rows Kimi-K2 3164 -> 3004 and GLM-4.5 827 -> 721,
// at 36 DeepSeek-V3 2170 -> 2027, at 75 DeepSeek-V3 2445 -> 2331, Kimi-K2 3642 -> 3440 and GLM-4.5
// 983 -> 865; with Zipf(1.2) routing at 34 rows Kimi-K2 2722 -> 2665 and GLM-4.5 748 -> 668, at 72
// DeepSeek-V3 2411 -> 2327. At 81 and 83 rows DeepSeek-V3 2462 -> 2486 and Kimi-K2 3688 -> 3692
// (GLM-4.5 gains up to 115), at 125 to 256 the block kernels lead by up to 4 % (two thirds of the
// global -> LDS bytes per product). Block tiles of 64 rows, three workgroups per CU, were 1 to 2 %
// faster up to 40 rows under even routing (Kimi-K2 34 rows 2950), but experts of many such
// tiles under Zipf routing cost more than the block kernels' (Kimi-K2 34 rows 2826, DeepSeek-V3 36
// rows 1995 against 1940), and the host does not know the routing.
constexpr int kMidTileRows = 64;
constexpr int kMidTallRows = 128;
constexpr int kMidTallMaxRows = 76;
// Work items from which they run 16-row tiles (four per CU; see mid_rows), and 32-row tiles and
// small layers (two per CU).
constexpr long kMidMinItems16 = 1024;
constexpr long kMidMinItems = 512;

// Compute units of the current device (cached per device; 256 on MI355X), for
// persistent grids of one workgroup per CU.
inline int device_cu_count() {
  constexpr int kMaxDev = 64;
  static int cached[kMaxDev];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDev) return 256;
  int n = __atomic_load_n(&cached[dev], __ATOMIC_RELAXED);
  if (n <= 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    __atomic_store_n(&cached[dev], n, __ATOMIC_RELAXED);
  }
  return n;
}

// Tile list written by the mapping's scan kernel from the expert counts
// (tiles == nullptr: none). Row tiles stay inside one block; block tiles
// (span = 1) run across an expert's blocks and carry seg = (first tile of the
// expert, its tile count). Shared-expert tiles follow the routed ones.
// A tile is {expert, first slot, rows, first hq / y row}. With compact = 0 the
// rows are the slots themselves; with compact = 1 the routed rows are packed
// expert after expert (expert e's i-th slot is row sum_{e' < e} count_e' + i),
// the shared expert j's token t is row row_shared + j * T + t, and inv_pos
// receives these rows instead of slots.
struct TileOut {
  int4* tiles;
  int2* seg;
  int32_t* num_tiles;
  int max_tiles;
  int mt;
  int span;
  int n_shared;
  int compact;
  long row_shared;
};

// The pre-MoE RMSNorm of the layer's rows (with gamma set): v = x, or bf16(x +
// residual) written to res_out as the next residual stream; the rows normalized
// over their first ha columns.
struct NormRide {
  const uint16_t* res;
  const float* gamma;
  uint16_t* res_out;
  int ha;
  float eps;
};

// Up to this many tokens the norm rides in the router logits launch: every
// workgroup of that launch reads the token rows and computes their norm factors
// itself (at most 16384 columns).
constexpr int kNormRideT = 4;
constexpr int kNormRideMaxH = 16384;

// Work that router_logits_topk may fold into its launches for the layer: the
// quantization of x into xq / xs (when xq is set: 1x128 fp8 codes and fp32 scales,
// or with quant_mx MXFP8 codes and E8M0 scale bytes) and blockwise_mapping of the
// ids it selects (when tpid is set; ids only, no padding mask, inv_pos = inv,
// workspace map_ws, tile list `to`). With norm.gamma set, x is normalized first:
// inside the logits launch where it can ride (then the quantization rides too),
// otherwise by rms_norm_quant into xn (its codes land in xq / xs), which the router then
// reads. On return quant_done / map_done say which it did; the
// caller runs the rest itself (from xn when the norm was requested).
struct RouterFuse {
  uint8_t* xq;
  void* xs;
  int quant_mx;
  NormRide norm;
  void* xn;
  int B, N;
  int32_t *tpid, *b2e, *cond, *counts, *inv;
  void* map_ws;
  size_t map_ws_bytes;
  TileOut to;
  bool quant_done, map_done;
};

// moe_rms_norm_quant, or with mx the same pass with MXFP8 codes in q and E8M0 scale bytes in s.
int rms_norm_quant(const void* x_bf16, const void* residual_bf16, const float* gamma, int T, int H,
                   int hidden_actual, float eps, void* xn_bf16, void* residual_out_bf16, uint8_t* q,
                   void* s, bool mx, void* stream);

// moe_router_logits followed by moe_router_topk (no affinities output), with the
// split-K reduce folded into the top-k kernel; for callers that already checked
// the arguments of both.
int router_logits_topk(const void* x_bf16, const void* w_bf16, const float* bias, int T, int H,
                       int E, float* logits, void* workspace, size_t workspace_bytes,
                       const float* corr_bias, int K, int order, int scoring, int n_group,
                       int topk_group, int renorm, float renorm_eps, float routed_scale,
                       int32_t* ids, float* weights, void* stream, RouterFuse* fuse = nullptr);

// moe_expert_gate_up for the layer, whose tiles its own mapping wrote: at one token
// every slot of a tile holds token 0, and the kernel loads no token ids.
int layer_gate_up(const uint8_t* xq, const float* xs, int T, int H, int I, int E, const uint8_t* w13,
                  const float* w13_scale, const uint8_t* w13_shared, const float* w13_shared_scale,
                  int n_shared, const int32_t* tpid, int NB, const int32_t* tiles,
                  const int32_t* num_tiles, int max_tiles, int mt, uint8_t* hq, float* hs,
                  void* stream);

// moe_expert_gate_up_mx / moe_expert_down_mx for the layer, whose tiles its own
// mapping wrote: at one token (one row per tile, token 0) the MXFP4 GEMMs with K =
// 3072 load each wave's fragments for the whole K into registers at once.
int layer_gate_up_mx(const uint8_t* xq, const uint8_t* xs, int T, int H, int I, int E, int wfmt,
                     const uint8_t* w13, const uint8_t* w13_scale, const float* b13,
                     const uint8_t* w13_shared, const uint8_t* w13_shared_scale,
                     const float* b13_shared, int n_shared, const int32_t* token_position_to_id,
                     int NB, const int32_t* tiles, const int32_t* num_tiles, int max_tiles, int mt,
                     int act, float gate_lo, float gate_hi, float up_lo, float up_hi, uint8_t* hq,
                     uint8_t* hs, void* stream);
int layer_down_mx(const uint8_t* hq, const uint8_t* hs, int T, int H, int I, int E, int wfmt,
                  const uint8_t* w2, const uint8_t* w2_scale, const float* b2,
                  const uint8_t* w2_shared, const uint8_t* w2_shared_scale, const float* b2_shared,
                  int n_shared, int NB, const int32_t* tiles, const int32_t* num_tiles,
                  int max_tiles, int mt, void* y_bf16, void* stream);

// moe_expert_down_mx followed by moe_combine (no shared experts) in one launch for the
// layer at one token with MXFP4 w2 and I = 3072 (K <= 8 pairs; ids, inv and weights of
// the token's pairs, inv the compact rows of hq): the same output bits without the y
// rows. *done says whether it ran; otherwise the caller runs both.
int layer_down_combine_mx(const uint8_t* hq, const uint8_t* hs, int T, int H, int I, int E, int K,
                          int wfmt, const uint8_t* w2, const uint8_t* w2_scale, const float* b2,
                          const int32_t* ids, const int32_t* inv, const float* weights,
                          void* out_bf16, void* stream, bool* done);

// Most block tiles of kMidTallRows rows that the layer's mapping writes (compact rows).
int mid_max_tiles(int T, int K, int E, int n_shared);

// Most block tiles of kMxBlockTileRows rows that the layer's mapping writes (compact rows).
int mx_block_max_tiles(int T, int K, int E);

// moe_blockwise_mapping plus an optional tile list (same checks and errors).
int blockwise_mapping(const int32_t* ids, const float* affinities, const uint8_t* padding_mask,
                      int T, int K, int E, int B, int N, int32_t* token_position_to_id,
                      int32_t* block_to_expert, int32_t* conditions, int32_t* expert_counts,
                      int32_t* inv_pos, float* affinities_masked, void* workspace,
                      size_t workspace_bytes, const TileOut& to, void* stream);

}  // namespace moe

#define MOE_API_BEGIN(name)   \
  const char* _moe_fn = name; \
  moe::clear_error();

#define MOE_CHECK_ARG(cond, ...)            \
  do {                                      \
    if (!(cond)) {                          \
      moe::set_error(_moe_fn, __VA_ARGS__); \
      return MOE_ERR_ARG;                   \
    }                                       \
  } while (0)

#define MOE_CHECK_SUPPORTED(cond, ...)      \
  do {                                      \
    if (!(cond)) {                          \
      moe::set_error(_moe_fn, __VA_ARGS__); \
      return MOE_ERR_UNSUPPORTED;           \
    }                                       \
  } while (0)

#define MOE_CHECK_HIP(expr)                                                              \
  do {                                                                                   \
    hipError_t _e = (expr);                                                              \
    if (_e != hipSuccess) {                                                              \
      moe::set_error(_moe_fn, "%s failed: %s", #expr, hipGetErrorString(_e));            \
      return MOE_ERR_HIP;                                                                \
    }                                                                                    \
  } while (0)

#define MOE_API_END()                                                                    \
  do {                                                                                   \
    hipError_t _e = hipGetLastError();                                                   \
    if (_e != hipSuccess) {                                                              \
      moe::set_error(_moe_fn, "kernel launch failed: %s", hipGetErrorString(_e));        \
      return MOE_ERR_HIP;                                                                \
    }                                                                                    \
    return MOE_OK;                                                                       \
  } while (0)
