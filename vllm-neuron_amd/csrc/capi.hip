// C-ABI glue: error strings, version, and the whole-layer forward that chains
// the kernels on one stream with a caller-provided workspace.
#include <stdarg.h>
#include <stdio.h>

#include <mutex>

#include "gemm_mid.h"
#include "gemm_mx.h"
#include "moe_common.h"
#include "moe_internal.h"

namespace moe {

static thread_local char g_err[1024] = {0};

void set_error(const char* fn, const char* fmt, ...) {
  int n = snprintf(g_err, sizeof(g_err), "%s: ", fn);
  if (n < 0 || n >= (int)sizeof(g_err)) return;
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err + n, sizeof(g_err) - n, fmt, ap);
  va_end(ap);
}

void clear_error() { g_err[0] = 0; }

// Rows per row tile (see use_block for the measurements): 16 up to 4 routed rows per expert on
// average, 32 up to 24 (layer_rows and mx_layer_rows raise some of them to 64), 64 up to 48, else
// 128. Above 32 rows the fp8 layer runs block tiles, the MX layer where it has items for them.
static int choose_mt(int T, int K, int E) {
  long avg = ((long)T * std::min(K, E) + E - 1) / E;
  if (avg <= 4) return 16;
  if (avg <= 24) return 32;
  if (avg <= 48) return 64;
  return 128;
}

// The MX row-tile kernels stop at 64-row tiles: at 128 rows the MXFP4 form of the
// kernel spills registers, and larger tiles only save L2 reads of the weights.
static int choose_mt_mx(int T, int K, int E) { return std::min(choose_mt(T, K, E), 64); }

struct LayerWs {
  uint16_t* xn;  // normalized rows (bf16), when the layer normalizes
  float* logits;
  void* router_ws;
  size_t router_ws_bytes;
  int32_t* ids;
  float* weights;
  int32_t* tpid;
  int32_t* b2e;
  int32_t* cond;
  int32_t* counts;
  int32_t* inv;
  void* map_ws;
  size_t map_ws_bytes;
  uint8_t* xq;
  float* xs;
  int32_t* tiles;
  int32_t* num_tiles;
  uint8_t* hq;
  float* hs;
  uint16_t* y;
  int32_t* btiles;
  int32_t* bnum;
  size_t bytes;
};

// Block tiles (of whole experts, in XCD ranges) take over from row tiles above 32 rows per expert on
// average: on the mid-size kernels up to kMidTallMaxRows, else on the 256x256 block kernels.
// Expert GEMM time (gate_up + down) on the DeepSeek-V3 layer by rows per expert, ms, ring kernels
// on row tiles of 16 / 32 / 64 rows against the block kernels: 4 rows 1.81 / 1.81 / 1.93 vs 2.05; 8:
// 1.95 / 1.92 / 2.08 vs 2.15; 16: 2.30 / 2.03 / 2.13 vs 2.29; 24: 2.78 / 2.11 / 2.19 vs 2.37; 32:
// 3.32 / 2.36 / 2.28 vs 2.42; 48: - / 2.95 / 2.47 vs 2.51; 64: - / 3.58 / 3.01 vs 2.60. On the Kimi-K2
// layer at 42.7 rows the block kernels led (3.90 against 3.95-4.00 ms), hence 32. The
// figures predate the mid-size kernels, which now run most of these tiles on both sides of the line.
static bool use_block(int T, int K, int E) {
  return ((long)T * std::min(K, E) + E - 1) / E > 32;
}

static inline size_t al(size_t x) { return (x + 255) & ~(size_t)255; }

// Routed rows held by the layer's hq / y buffers: every routed (token, expert)
// pair has a row (packed expert by expert), then n_shared * T shared rows.
static inline long routed_rows(int T, int K, int E) { return (long)T * std::min(K, E); }

// Carves the workspace (base may be null to size it).
static LayerWs carve(char* base, int T, int H, int I, int E, int K, int n_sh, int B, bool norm) {
  LayerWs w{};
  const int N = moe_num_blocks(T, K, E, B);
  const long NB = (long)N * B;
  const long P = routed_rows(T, K, E) + (long)n_sh * T;
  // tile list sized for the smaller of the two layers' tile heights (more tiles)
  const int mt = choose_mt_mx(T, K, E);
  const int max_tiles = moe_max_tiles(T, K, E, N, B, n_sh, mt);
  size_t off = 0;
  auto take = [&](size_t bytes) -> char* {
    char* p = base ? base + off : nullptr;
    off += al(bytes);
    return p;
  };
  if (norm) w.xn = (uint16_t*)take((size_t)T * H * 2);
  w.logits = (float*)take((size_t)T * E * 4);
  w.router_ws_bytes = moe_router_logits_workspace_bytes(T, H, E);
  w.router_ws = take(w.router_ws_bytes);
  w.ids = (int32_t*)take((size_t)T * K * 4);
  w.weights = (float*)take((size_t)T * K * 4);
  w.tpid = (int32_t*)take((size_t)NB * 4);
  w.b2e = (int32_t*)take((size_t)N * 4);
  w.cond = (int32_t*)take((size_t)N * 4);
  w.counts = (int32_t*)take((size_t)E * 4);
  w.inv = (int32_t*)take((size_t)T * K * 4);
  w.map_ws_bytes = moe_mapping_workspace_bytes(T, E);
  w.map_ws = take(w.map_ws_bytes);
  w.xq = (uint8_t*)take((size_t)T * H);
  w.xs = (float*)take((size_t)T * (H / 128) * 4);
  w.tiles = (int32_t*)take((size_t)max_tiles * 16);
  w.num_tiles = (int32_t*)take(16);
  w.hq = (uint8_t*)take((size_t)P * I);
  w.hs = (float*)take((size_t)P * (I / 128) * 4);
  w.y = (uint16_t*)take((size_t)P * H * 2);
  if (use_block(T, K, E)) {
    const int mbt = moe_max_block_tiles(T, K, E, N, B, n_sh);
    w.btiles = (int32_t*)take((size_t)mbt * 24);
    w.bnum = (int32_t*)take(MOE_BLOCK_TILES_HEADER * 4);  // count + XCD ranges
  }
  w.bytes = off;
  return w;
}

}  // namespace moe

using namespace moe;

extern "C" int moe_abi_version(void) { return MOE_FP8_ABI_VERSION; }

extern "C" const char* moe_last_error(void) { return g_err; }

extern "C" size_t moe_layer_workspace_bytes(int T, int H, int I, int E, int K, int n_shared, int B,
                                            int norm) {
  if (T <= 0 || H <= 0 || I <= 0 || E <= 0 || K <= 0 || n_shared < 0 || B <= 0) return 0;
  return carve(nullptr, T, H, I, E, K, n_shared, B, norm != 0).bytes;
}

// RouterFuse for the layer's mapping (no quantization).
static RouterFuse map_fuse(const LayerWs& w, int B, int N, const TileOut& to) {
  RouterFuse fz{};
  fz.B = B;
  fz.N = N;
  fz.tpid = w.tpid;
  fz.b2e = w.b2e;
  fz.cond = w.cond;
  fz.counts = w.counts;
  fz.inv = w.inv;
  fz.map_ws = w.map_ws;
  fz.map_ws_bytes = w.map_ws_bytes;
  fz.to = to;
  return fz;
}

// Rows per tile of the fp8 layer's row tiles; mid_ok: the mid-size kernels fit its products.
static int layer_rows(int T, int H, int I, int E, int K, int n_shared, int B, bool mid_ok) {
  const int mt = choose_mt(T, K, E);
  if (!mid_ok || mt != 32) return mt;
  // Of 5 to 24 rows per expert, 64-row tiles keep nearly every expert in one tile, where both
  // products then have enough items. With few items of down, its 32-row tiles stay on the ring
  // kernels: 8 experts of 4096 x 14336 (128 down items of K = 14336), 24 / 48 / 96 tokens, gate_up and
  // down on the ring 293 / 296 / 305, both on 64-row tiles 343 / 345 / 350, so 268 / 270 / 276 us.
  const int t64 = moe_max_tiles(T, K, E, moe_num_blocks(T, K, E, B), B, n_shared, kMidTileRows);
  return (long)t64 * std::min(I / 128, H / 256) >= kMidMinItems ? kMidTileRows : mt;
}

// Whether the fp8 layer runs the mid-size kernels on block tiles, where they fit.
static bool layer_mid(int T, int I, int E, int K, int n_shared) {
  return use_block(T, K, E) && routed_rows(T, K, E) <= kMidTallMaxRows * (long)E &&
         (long)mid_max_tiles(T, K, E, n_shared) * (I / 128) >= kMidMinItems;
}

extern "C" int moe_row_tile_kernels(int H, int I, int max_tiles, int mt) {
  if (H <= 0 || I <= 0 || max_tiles <= 0) return 0;
  MidArgs a{};
  a.H = H;
  a.I = I;
  int on_mid = 0;
  for (int kind = 0; kind < 2; ++kind)
    on_mid |= (mid_rows(kind, H, I, max_tiles, mt) && mid_fits(kind, a)) << kind;
  return on_mid;
}

extern "C" int moe_layer_tile_rows(int T, int H, int I, int E, int K, int n_shared, int B) {
  if (T <= 0 || H <= 0 || I <= 0 || E <= 0 || K <= 0 || n_shared < 0 || B <= 0) return 0;
  MidArgs a{};
  a.T = T;
  a.H = H;
  a.I = I;
  a.rows = routed_rows(T, K, E) + (long)n_shared * T;
  const bool mid_ok = mid_fits(0, a) && mid_fits(1, a);
  if (!use_block(T, K, E)) return layer_rows(T, H, I, E, K, n_shared, B, mid_ok);
  return mid_ok && layer_mid(T, I, E, K, n_shared) ? kMidTallRows : kBlockTileRows;
}

// The layer forward of both entry points: `workspace` is the caller's buffer or
// this device's static scratch. _moe_fn names the entry point in error messages.
static int layer_forward_impl(const char* _moe_fn, const void* x_bf16, const void* residual_bf16,
                              const float* gamma, float eps, int hidden_actual, int T, int H,
                              int I, int E, int K, int n_shared, const void* router_w_bf16,
                              const float* router_bias, const float* corr_bias, int order,
                              int scoring, int n_group, int topk_group, int renorm,
                              float renorm_eps, float routed_scale, const uint8_t* w13,
                              const float* w13_scale, const uint8_t* w2, const float* w2_scale,
                              const uint8_t* w13_shared, const float* w13_shared_scale,
                              const uint8_t* w2_shared, const float* w2_shared_scale, int B,
                              void* out_bf16, void* residual_out_bf16, int32_t* ids_out,
                              float* weights_out, float* logits_out, void* workspace,
                              size_t workspace_bytes, void* stream) {
  MOE_CHECK_ARG(x_bf16 && router_w_bf16 && w13 && w13_scale && w2 && w2_scale && out_bf16 && workspace,
                "null pointer argument");
  MOE_CHECK_ARG(T > 0 && E > 0 && K > 0 && K <= E && B > 0 && n_shared >= 0,
                "bad sizes T=%d E=%d K=%d B=%d", T, E, K, B);
  MOE_CHECK_ARG(H % 256 == 0 && I % 128 == 0, "H must be a multiple of 256 and I of 128");
  MOE_CHECK_ARG((residual_bf16 == nullptr) == (residual_out_bf16 == nullptr),
                "residual and residual_out must be given together");
  MOE_CHECK_ARG(gamma != nullptr || residual_bf16 == nullptr,
                "the residual add is fused into the norm: residual needs gamma");
  const bool norm = gamma != nullptr;
  const size_t need = moe_layer_workspace_bytes(T, H, I, E, K, n_shared, B, norm);
  MOE_CHECK_ARG(workspace_bytes >= need, "workspace too small: need %zu bytes, got %zu", need,
                workspace_bytes);
  MOE_CHECK_ARG(((uintptr_t)workspace & 255) == 0, "workspace must be 256-byte aligned");
  LayerWs w = carve((char*)workspace, T, H, I, E, K, n_shared, B, norm);
  const int N = moe_num_blocks(T, K, E, B);
  const long NB = (long)N * B;
  const long R = routed_rows(T, K, E);
  MOE_CHECK_SUPPORTED(NB + (long)n_shared * T < (1L << 31), "too many slots");
  // operands of the mid-size kernels
  MidArgs mg{}, md{};
  mg.a = w.xq;
  mg.as = w.xs;
  mg.w = w13;
  mg.ws = w13_scale;
  mg.wsh = w13_shared;
  mg.wssh = w13_shared_scale;
  mg.tpid = w.tpid;
  mg.tiles = (const int4*)w.tiles;
  mg.seg = (const int2*)w.btiles;
  mg.num_tiles = w.bnum;
  mg.hq = w.hq;
  mg.hs = w.hs;
  mg.T = T;
  mg.H = H;
  mg.I = I;
  mg.E = E;
  mg.nsh = n_shared;
  mg.NB = NB;
  mg.rows = R + (long)n_shared * T;
  md = mg;
  md.a = w.hq;
  md.as = w.hs;
  md.w = w2;
  md.ws = w2_scale;
  md.wsh = w2_shared;
  md.wssh = w2_shared_scale;
  md.y = w.y;
  const bool mid_ok = mid_fits(0, mg) && mid_fits(1, md);
  const int mt = layer_rows(T, H, I, E, K, n_shared, B, mid_ok);
  const int max_tiles = moe_max_tiles(T, K, E, N, B, n_shared, mt);
  float* logits = logits_out ? logits_out : w.logits;
  int32_t* ids = ids_out ? ids_out : w.ids;
  float* wts = weights_out ? weights_out : w.weights;

  char saved[1024];
  int rc;
#define MOE_STEP(call)                                         \
  rc = (call);                                                 \
  if (rc != MOE_OK) {                                          \
    snprintf(saved, sizeof(saved), "%s", moe_last_error());    \
    moe::set_error(_moe_fn, "%s", saved);                      \
    return rc;                                                 \
  }
  // The mapping also writes the expert tile list, from the counts.
  const bool block = use_block(T, K, E);
  const int mbt = block ? moe_max_block_tiles(T, K, E, N, B, n_shared) : 0;
  // Above 32 and up to kMidTallMaxRows rows per expert on average, 128-row block tiles: their
  // list goes into the row-tile list's room (sized for 64-row tiles), its segments (8 bytes each)
  // into the block tiles' (24 bytes each).
  const int mmt = block ? mid_max_tiles(T, K, E, n_shared) : 0;
  const bool mid = mid_ok && layer_mid(T, I, E, K, n_shared) &&
                   mmt <= moe_max_tiles(T, K, E, N, B, n_shared, choose_mt_mx(T, K, E)) && mmt <= 3L * mbt;
  TileOut to{};
  if (mid) {
    to.tiles = (int4*)w.tiles;
    to.seg = (int2*)w.btiles;
    to.num_tiles = w.bnum;
    to.max_tiles = mmt;
    to.mt = kMidTallRows;
    to.span = 1;
  } else if (block) {
    to.tiles = (int4*)w.btiles;
    to.seg = (int2*)(w.btiles + 4 * (size_t)mbt);
    to.num_tiles = w.bnum;
    to.max_tiles = mbt;
    to.mt = kBlockTileRows;
    to.span = 1;
  } else {
    to.tiles = (int4*)w.tiles;
    to.num_tiles = w.num_tiles;
    to.max_tiles = max_tiles;
    to.mt = mt;
  }
  to.n_shared = n_shared;
  to.compact = 1;  // hq / y hold only the routed and shared rows
  to.row_shared = R;
  // Pre-MoE RMSNorm (with the residual add) and the 1x128 quantization of the
  // normalized rows: up to a few tokens inside the logits launch, else in one pass
  // before it (router_logits_topk). Decode sizes: the quantization rides in the
  // logits launch and the mapping ends the top-k launch (router_logits_topk says
  // which it did).
  RouterFuse fz = map_fuse(w, B, N, to);
  fz.xq = w.xq;
  fz.xs = w.xs;
  if (norm) {
    fz.norm = NormRide{(const uint16_t*)residual_bf16, gamma, (uint16_t*)residual_out_bf16,
                       hidden_actual > 0 ? hidden_actual : H, eps};
    fz.xn = w.xn;
  }
  MOE_STEP(router_logits_topk(x_bf16, router_w_bf16, router_bias, T, H, E, logits, w.router_ws,
                              w.router_ws_bytes, corr_bias, K, order, scoring, n_group, topk_group,
                              renorm, renorm_eps, routed_scale, ids, wts, stream, &fz));
  if (!fz.map_done)
    MOE_STEP(blockwise_mapping(ids, nullptr, nullptr, T, K, E, B, N, w.tpid, w.b2e, w.cond, w.counts,
                               w.inv, nullptr, w.map_ws, w.map_ws_bytes, to, stream));
  // (with the norm the quantization is always done: in the logits launch or by the norm)
  if (!fz.quant_done) MOE_STEP(moe_act_quant_1x128(x_bf16, T, H, w.xq, w.xs, stream));
  if (mid) {
    MOE_CHECK_ARG(n_shared == 0 || (w13_shared && w13_shared_scale && w2_shared && w2_shared_scale),
                  "shared weights missing");
    launch_mid(0, mg, mmt, (hipStream_t)stream);
    launch_mid(1, md, mmt, (hipStream_t)stream);
  } else if (block) {
    MOE_STEP(moe_expert_gate_up_block(w.xq, w.xs, T, H, I, E, w13, w13_scale, nullptr, w13_shared,
                                      w13_shared_scale, nullptr, n_shared, w.tpid, (int)NB, w.btiles,
                                      w.bnum, mbt, w.hq, w.hs, stream));
    MOE_STEP(moe_expert_down_block(w.hq, w.hs, T, H, I, E, w2, w2_scale, nullptr, w2_shared,
                                   w2_shared_scale, nullptr, n_shared, (int)NB, w.btiles, w.bnum, mbt,
                                   w.y, stream));
  } else {
    MOE_STEP(layer_gate_up(w.xq, w.xs, T, H, I, E, w13, w13_scale, w13_shared, w13_shared_scale,
                           n_shared, w.tpid, (int)NB, w.tiles, w.num_tiles, max_tiles, mt, w.hq, w.hs,
                           stream));
    MOE_STEP(moe_expert_down(w.hq, w.hs, T, H, I, E, w2, w2_scale, nullptr, w2_shared,
                             w2_shared_scale, nullptr, n_shared, (int)NB, w.tiles, w.num_tiles,
                             max_tiles, mt, w.y,
                             stream));
  }
  MOE_STEP(moe_combine(w.y, w.inv, wts, K, T, H, (int)R, n_shared, out_bf16, stream));
#undef MOE_STEP
  return MOE_OK;
}

extern "C" int moe_layer_forward(const void* x_bf16, const void* residual_bf16,
                                 const float* gamma, float eps, int hidden_actual, int T, int H,
                                 int I, int E, int K, int n_shared, const void* router_w_bf16,
                                 const float* router_bias, const float* corr_bias, int order,
                                 int scoring, int n_group, int topk_group, int renorm,
                                 float renorm_eps, float routed_scale, const uint8_t* w13,
                                 const float* w13_scale, const uint8_t* w2, const float* w2_scale,
                                 const uint8_t* w13_shared, const float* w13_shared_scale,
                                 const uint8_t* w2_shared, const float* w2_shared_scale, int B,
                                 void* out_bf16, void* residual_out_bf16, int32_t* ids_out,
                                 float* weights_out, float* logits_out, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  MOE_API_BEGIN("moe_layer_forward");
  return layer_forward_impl(_moe_fn, x_bf16, residual_bf16, gamma, eps, hidden_actual, T, H, I, E,
                            K, n_shared, router_w_bf16, router_bias, corr_bias, order, scoring,
                            n_group, topk_group, renorm, renorm_eps, routed_scale, w13, w13_scale,
                            w2, w2_scale, w13_shared, w13_shared_scale, w2_shared,
                            w2_shared_scale, B, out_bf16, residual_out_bf16, ids_out, weights_out,
                            logits_out, workspace, workspace_bytes, stream);
}

// ---------------------------------------------------------------------------
// Allocation-free layer forward. Its workspace is `scratch`, one static array per
// GPU that the code object's loader places in device memory and that lives until
// the process ends. In host code `scratch` names a host-side shadow, not device
// memory, so its device address is looked up once per device with
// hipGetSymbolAddress (with that device current) and only that address is handed
// to kernels. Calls on one GPU share the array: they must not overlap (same
// stream or otherwise ordered), and nothing in it has to start at zero (every
// kernel of the layer writes what it later reads; the mapping clears its own
// status word).
// ---------------------------------------------------------------------------
static __device__ __align__(256) uint8_t scratch[MOE_NOALLOC_SCRATCH_BYTES];

namespace moe {

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_dev[kMaxDevices];

// Device address of this device's `scratch` (looked up on the first call per device).
static int scratch_address(const char* _moe_fn, void** out) {
  int dev = -1;
  MOE_CHECK_HIP(hipGetDevice(&dev));
  MOE_CHECK_SUPPORTED(dev >= 0 && dev < kMaxDevices, "device %d beyond %d", dev, kMaxDevices);
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_dev[dev] == nullptr) {
    void* p = nullptr;
    MOE_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    MOE_CHECK_ARG(p != nullptr && ((uintptr_t)p & 255) == 0, "bad scratch address");
    g_scratch_dev[dev] = p;
  }
  *out = g_scratch_dev[dev];
  return MOE_OK;
}

}  // namespace moe

extern "C" int moe_layer_forward_noalloc(
    const void* x_bf16, const void* residual_bf16, const float* gamma, float eps,
    int hidden_actual, int T, int H, int I, int E, int K, int n_shared, const void* router_w_bf16,
    const float* router_bias, const float* corr_bias, int order, int scoring, int n_group,
    int topk_group, int renorm, float renorm_eps, float routed_scale, const uint8_t* w13,
    const float* w13_scale, const uint8_t* w2, const float* w2_scale, const uint8_t* w13_shared,
    const float* w13_shared_scale, const uint8_t* w2_shared, const float* w2_shared_scale, int B,
    void* out_bf16, void* residual_out_bf16, int32_t* ids_out, float* weights_out,
    float* logits_out, void* stream) {
  MOE_API_BEGIN("moe_layer_forward_noalloc");
  MOE_CHECK_ARG(T > 0 && H > 0 && I > 0 && E > 0 && K > 0 && B > 0 && n_shared >= 0,
                "bad sizes T=%d H=%d I=%d E=%d K=%d B=%d", T, H, I, E, K, B);
  const size_t need = moe_layer_workspace_bytes(T, H, I, E, K, n_shared, B, gamma != nullptr);
  MOE_CHECK_SUPPORTED(need <= (size_t)MOE_NOALLOC_SCRATCH_BYTES,
                      "this layer call needs %zu bytes of scratch; the static scratch holds %zu "
                      "(use moe_layer_forward with a workspace)",
                      need, (size_t)MOE_NOALLOC_SCRATCH_BYTES);
  void* ws = nullptr;
  const int rc = scratch_address(_moe_fn, &ws);
  if (rc != MOE_OK) return rc;
  return layer_forward_impl(_moe_fn, x_bf16, residual_bf16, gamma, eps, hidden_actual, T, H, I, E,
                            K, n_shared, router_w_bf16, router_bias, corr_bias, order, scoring,
                            n_group, topk_group, renorm, renorm_eps, routed_scale, w13, w13_scale,
                            w2, w2_scale, w13_shared, w13_shared_scale, w2_shared,
                            w2_shared_scale, B, out_bf16, residual_out_bf16, ids_out, weights_out,
                            logits_out, ws, (size_t)MOE_NOALLOC_SCRATCH_BYTES, stream);
}

// Rows per tile of the MX layer's row tiles; block_ok: the block kernels fit its products.
static int mx_layer_rows(int T, int H, int I, int E, int K, int B, bool block_ok) {
  const int mt = choose_mt_mx(T, K, E), N = moe_num_blocks(T, K, E, B);
  if (!block_ok || mt != 32) return mt;
  // Of 5 to 24 rows per expert, 64-row tiles keep nearly every expert in one tile: above 16 rows
  // where the block kernels run both products on them, or gate_up on them and down on neither
  // height (64 experts of 1024 x 2048, 20 rows: 87 -> 75 us), below that where they have 1024 items in
  // both, two rounds (GPT-OSS-120B under Zipf routing, 8 / 12 / 16 rows 191 / 243 / 263 -> 179 / 214 /
  // 230 us, even routing within 1 %). In one round the tallest tile sets the time, which shows under
  // skewed routing (64 experts of 2048 x 1024 under Zipf routing, 4 to 6 rows: 43.5 to 45.2 at 32 rows,
  // 46.9 to 49.4 us at 64). They lose too with down on the ring kernels (160 experts of 512 x 1024, 5 /
  // 8 rows: 57.2 / 65.5 at 32 rows, 62.9 / 69.7 us at 64), and where the ring keeps gate_up at 32 rows
  // (GPT-OSS-20B, 33 / 64 / 80 / 135 tokens 117 / 120 / 114 / 118 at 32 rows, 125 / 127 / 128 / 130 us
  // at 64).
  const int t32 = moe_max_tiles(T, K, E, N, B, 0, 32), t64 = moe_max_tiles(T, K, E, N, B, 0, 64);
  auto on_block = [&](int kind, int rows) {
    return mx_rows_on_block(kind, H, I, E, rows == 32 ? t32 : t64, rows);
  };
  if (!on_block(0, 32) || !on_block(0, 64)) return 32;
  const bool many = routed_rows(T, K, E) > 16L * E || (long)t64 * std::min(I / 128, H / 256) >= 2 * kMidMinItems;
  const bool tall = many && (on_block(1, 64) || !on_block(1, 32));
  return tall ? 64 : 32;
}

// Whether the MXFP4 layer runs block tiles: above 32 rows per expert, where 64-row tiles are more
// than one round of the ring kernels' one workgroup per CU in one product (from 320 items, counted
// with a remainder tile for each expert). In one round a taller tile is only a longer chain. Layer,
// 64-row tiles on the ring -> block tiles, us: 4 experts of 512 x 512 at 64 / 100 / 256 rows per
// expert 36.9 / 37.2 / 43.3 -> 36.7 / 41.1 / 47.2; 8 of 1024 x 1024 at 80 / 200 / 256 (264 and 320
// items) 50.6 / 54.0 / 65.7 -> 53.3 / 54.3 / 56.9; 4 of 3072 x 3072 at 128 / 150 (288 and 336 items)
// 71.3 / 98.7 -> 80.2 / 74.5. Up to 40 rows an expert is mostly one tile in both, and block tiles gain
// under even routing (16 of 512 x 512, 36 rows: 42.8 -> 37.6) but lose under Zipf routing (43.5 ->
// 47.3; 8 of 1024 x 1024, 33 rows: 43.4 -> 49.4), which the host does not know.
constexpr long kMxBlockMinItems = 320;
static bool mx_layer_block(int T, int H, int I, int E, int K, int B) {
  if (!use_block(T, K, E)) return false;
  const long R = routed_rows(T, K, E), tiles = (R + std::min(64, B) - 1) / std::min(64, B) + E;
  return tiles * std::max(I / 128, H / 256) >= kMxBlockMinItems;
}

extern "C" int moe_layer_mx_tile_rows(int T, int H, int I, int E, int K, int B) {
  if (T <= 0 || H <= 0 || I <= 0 || E <= 0 || K <= 0 || B <= 0) return 0;
  MxArgs a{};
  a.T = T;
  a.H = H;
  a.I = I;
  a.rows = routed_rows(T, K, E);
  const bool block_ok = mx_block_fits(0, a) && mx_block_fits(1, a);
  return block_ok && mx_layer_block(T, H, I, E, K, B) ? kMxBlockTileRows
                                                      : mx_layer_rows(T, H, I, E, K, B, block_ok);
}

// ---------------------------------------------------------------------------
// The layer with MX experts (GPT-OSS): [residual add ->] [RMSNorm ->] router ->
// top-k -> mapping (compact rows) -> MXFP8 quantization -> MX gate_up (bias,
// clamps, activation) -> MX down (bias) -> combine. Same workspace as
// moe_layer_forward without shared experts (the MX scale bytes take the room of
// the 1x128 fp32 scales).
// ---------------------------------------------------------------------------
extern "C" int moe_layer_forward_mx(
    const void* x_bf16, const void* residual_bf16, const float* gamma, float eps,
    int hidden_actual, int T, int H, int I, int E, int K, const void* router_w_bf16,
    const float* router_bias, int order, int scoring, int renorm, float renorm_eps,
    float routed_scale, int wfmt, const uint8_t* w13, const uint8_t* w13_scale, const float* b13,
    const uint8_t* w2, const uint8_t* w2_scale, const float* b2, int act, float gate_lo,
    float gate_hi, float up_lo, float up_hi, int B, void* out_bf16, void* residual_out_bf16,
    int32_t* ids_out, float* weights_out, float* logits_out, void* workspace,
    size_t workspace_bytes, void* stream) {
  MOE_API_BEGIN("moe_layer_forward_mx");
  MOE_CHECK_ARG(x_bf16 && router_w_bf16 && w13 && w13_scale && w2 && w2_scale && out_bf16 && workspace,
                "null pointer argument");
  MOE_CHECK_ARG(T > 0 && E > 0 && K > 0 && K <= E && B > 0, "bad sizes T=%d E=%d K=%d B=%d", T, E,
                K, B);
  MOE_CHECK_ARG(H % 256 == 0 && I % 128 == 0, "H must be a multiple of 256 and I of 128 (pad them)");
  MOE_CHECK_ARG(order == MOE_ORDER_TOPK_ACT || order == MOE_ORDER_ACT_TOPK,
                "the MX layer routes with the TOPK_ACT or ACT_TOPK order");
  MOE_CHECK_ARG((residual_bf16 == nullptr) == (residual_out_bf16 == nullptr),
                "residual and residual_out must be given together");
  MOE_CHECK_ARG(gamma != nullptr || residual_bf16 == nullptr,
                "the residual add is fused into the norm: residual needs gamma");
  const bool norm = gamma != nullptr;
  const size_t need = moe_layer_workspace_bytes(T, H, I, E, K, 0, B, norm);
  MOE_CHECK_ARG(workspace_bytes >= need, "workspace too small: need %zu bytes, got %zu", need,
                workspace_bytes);
  MOE_CHECK_ARG(((uintptr_t)workspace & 255) == 0, "workspace must be 256-byte aligned");
  LayerWs w = carve((char*)workspace, T, H, I, E, K, 0, B, norm);
  const int N = moe_num_blocks(T, K, E, B);
  const long NB = (long)N * B;
  const long R = routed_rows(T, K, E);
  MOE_CHECK_SUPPORTED(NB < (1L << 31), "too many slots");
  // operands of the block kernels
  MxArgs bg{}, bd{};
  bg.a = w.xq;
  bg.as = (const uint8_t*)w.xs;
  bg.w = w13;
  bg.ws = w13_scale;
  bg.bias = b13;
  bg.tpid = w.tpid;
  bg.tiles = (const int4*)w.tiles;
  bg.seg = (const int2*)w.btiles;
  bg.num_tiles = w.bnum;
  bg.hq = w.hq;
  bg.hs = (uint8_t*)w.hs;
  bg.T = T;
  bg.H = H;
  bg.I = I;
  bg.E = E;
  bg.NB = NB;
  bg.rows = R;
  auto lim = [](float v, float dflt) { return v != v ? dflt : v; };  // NaN: no limit
  bg.act = act;
  bg.gate_lo = lim(gate_lo, -__builtin_inff());
  bg.gate_hi = lim(gate_hi, __builtin_inff());
  bg.up_lo = lim(up_lo, -__builtin_inff());
  bg.up_hi = lim(up_hi, __builtin_inff());
  bd = bg;
  bd.a = w.hq;
  bd.as = (const uint8_t*)w.hs;
  bd.w = w2;
  bd.ws = w2_scale;
  bd.bias = b2;
  bd.y = w.y;
  const bool block_ok = wfmt == MOE_MX_FP4 && (act == MOE_ACT_SILU || act == MOE_ACT_SWISH) &&
                        mx_block_fits(0, bg) && mx_block_fits(1, bd);
  const int mt = mx_layer_rows(T, H, I, E, K, B, block_ok);
  const int max_tiles = moe_max_tiles(T, K, E, N, B, 0, mt);
  float* logits = logits_out ? logits_out : w.logits;
  int32_t* ids = ids_out ? ids_out : w.ids;
  float* wts = weights_out ? weights_out : w.weights;
  uint8_t* xs = (uint8_t*)w.xs;  // T * H/32 bytes of E8M0 scales
  uint8_t* hs = (uint8_t*)w.hs;  // P * I/32 bytes

  char saved[1024];
  int rc;
#define MOE_STEP(call)                                         \
  rc = (call);                                                 \
  if (rc != MOE_OK) {                                          \
    snprintf(saved, sizeof(saved), "%s", moe_last_error());    \
    moe::set_error(_moe_fn, "%s", saved);                      \
    return rc;                                                 \
  }
  // Block tiles go into the row-tile list's room (at most R / 128 + E of them, which is no more
  // than the R / 64 + N row tiles it is sized for, N >= E), their segments (8 bytes each) into
  // the fp8 block tiles' (24 bytes for each of NB / 256 + E, NB >= R).
  const bool block = block_ok && mx_layer_block(T, H, I, E, K, B);
  const int mbt = block ? mx_block_max_tiles(T, K, E) : 0;
  TileOut to{};
  to.tiles = (int4*)w.tiles;
  if (block) {
    MOE_CHECK_ARG(mbt <= max_tiles && mbt <= 3 * moe_max_block_tiles(T, K, E, N, B, 0),
                  "tile list of %d block tiles does not fit the workspace", mbt);
    to.seg = (int2*)w.btiles;
    to.num_tiles = w.bnum;
    to.max_tiles = mbt;
    to.mt = kMxBlockTileRows;
    to.span = 1;
  } else {
    to.num_tiles = w.num_tiles;
    to.max_tiles = max_tiles;
    to.mt = mt;
  }
  to.compact = 1;
  to.row_shared = R;
  // Residual add + RMSNorm: up to a few tokens inside the logits launch, else in a
  // pass of its own before it, which quantizes the normalized rows too.
  // Decode sizes: the MXFP8 quantization rides in the logits launch and the
  // mapping ends the top-k launch (router_logits_topk says which it did).
  RouterFuse fz = map_fuse(w, B, N, to);
  fz.xq = w.xq;
  fz.xs = xs;
  fz.quant_mx = 1;
  if (norm) {
    fz.norm = NormRide{(const uint16_t*)residual_bf16, gamma, (uint16_t*)residual_out_bf16,
                       hidden_actual > 0 ? hidden_actual : H, eps};
    fz.xn = w.xn;
  }
  const void* xr = norm ? w.xn : x_bf16;  // what the router read, unless the norm rode
  MOE_STEP(router_logits_topk(x_bf16, router_w_bf16, router_bias, T, H, E, logits, w.router_ws,
                              w.router_ws_bytes, nullptr, K, order, scoring, 1, 1, renorm,
                              renorm_eps, routed_scale, ids, wts, stream, &fz));
  if (!fz.map_done)
    MOE_STEP(blockwise_mapping(ids, nullptr, nullptr, T, K, E, B, N, w.tpid, w.b2e, w.cond, w.counts,
                               w.inv, nullptr, w.map_ws, w.map_ws_bytes, to, stream));
  if (!fz.quant_done) MOE_STEP(moe_act_quant_mx(xr, T, H, w.xq, xs, stream));
  if (block) {
    launch_mx_block(0, bg, mbt, (hipStream_t)stream);
    launch_mx_block(1, bd, mbt, (hipStream_t)stream);
    MOE_STEP(moe_combine(w.y, w.inv, wts, K, T, H, (int)R, 0, out_bf16, stream));
    return MOE_OK;
  }
  MOE_STEP(layer_gate_up_mx(w.xq, xs, T, H, I, E, wfmt, w13, w13_scale, b13, nullptr, nullptr,
                            nullptr, 0, w.tpid, (int)NB, w.tiles, w.num_tiles, max_tiles, mt, act,
                            gate_lo, gate_hi, up_lo, up_hi, w.hq, hs, stream));
  bool fused = false;
  MOE_STEP(layer_down_combine_mx(w.hq, hs, T, H, I, E, K, wfmt, w2, w2_scale, b2, ids, w.inv, wts,
                                 out_bf16, stream, &fused));
  if (!fused) {
    MOE_STEP(layer_down_mx(w.hq, hs, T, H, I, E, wfmt, w2, w2_scale, b2, nullptr, nullptr, nullptr,
                           0, (int)NB, w.tiles, w.num_tiles, max_tiles, mt, w.y, stream));
    MOE_STEP(moe_combine(w.y, w.inv, wts, K, T, H, (int)R, 0, out_bf16, stream));
  }
#undef MOE_STEP
  return MOE_OK;
}
