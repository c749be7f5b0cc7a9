// MXFP4 expert GEMMs (GPT-OSS) on block tiles of up to 128 rows (the layer above 32 routed rows per
// expert, mx_layer_block) and on row tiles of 32 and 64 rows with enough items (the layer and the
// operators from 5 rows per expert, mx_rows_on_block). Same products, epilogue arithmetic and K
// order as the ring kernel (gemm_mx.hip), with two workgroups per CU, and block tiles tall enough
// that the matrix cores, not the weight stream of one 64-row tile, set the time.
//
//  * A workgroup of 4 waves computes up to 128 rows x 256 weight rows (gate_up: 128
//    gate rows + the matching 128 up rows; down: 256 outputs). A wave owns every row and
//    64 of the columns: MF = ceil(rows / 16) x 4 tiles of
//    v_mfma_scale_f32_16x16x128_f8f6f4, whose E8M0 operands apply every block scale. MXFP4
//    fragments take half the registers of the token fragments, so a wave holds its weight
//    fragments of a whole step (32 registers) and streams the token fragments from LDS; a
//    tile's work then follows its rows in steps of 16.
//  * 76.5 KB of LDS, so two workgroups share a CU (two waves per SIMD). They meet no
//    common barrier: one's fragment reads, waits, prologue and epilogue run under the
//    other's MFMAs.
//  * A step is 256 K values: 128 bytes of every weight row (whole cache lines) and two
//    128-byte pieces of every token row, by direct-to-LDS loads. The weight tile has one
//    32 KB buffer, free again once the fragments are in registers, so the next tile is on
//    its way for the rest of the step; each token half has its own 16 KB buffer.
//  * Weights carry the non-temporal hint: the scale lines (each read again for every 512 K
//    values) and the token rows then stay in L2. Bytes read beyond L2 by gate_up at 2048
//    tokens of GPT-OSS-120B: 1.58 -> 1.31 GB (1.28 GB of weights and scales); layer at 1100 /
//    2048 / 3200 tokens 480 / 545 / 640 -> 437 / 511 / 605 us, at 8192 and above unchanged.
//  * The scale bytes of 512 K values (16 per row) arrive with one 16-byte load per row
//    every second step.
//
// Measured, GPT-OSS-120B (kernel trace), against the ring kernels' 64-row tiles: gate_up 1408 -> 720
// us and down 629 -> 380 us at 8192 tokens (256 rows per expert), 516 -> 295 and 240 -> 157 us at 2048.
// At 8192 the MFMA pipes are busy 52 and 46 % of the time; gate_up without the in-loop loads takes
// 500 us, without the MFMAs 580 us (1.24 TFLOP, MFMA alone 280 us): both halves and their overlap. At
// 2048 26 and 23 %, with the weights read at 4.4 and 4.1 TB/s.
//
// Fragment layout as in gemm_mx.hip: lane l supplies row l % 16; with g = l / 16, the
// fp8 K values [16 g, +16) and [64 + 16 g, +16), the fp4 K values [32 g, +32) and the
// scale byte of K values [32 g, +32).
#include "gemm_mx.h"
#include "mapping.h"
#include "moe_common.h"
#include "moe_internal.h"

namespace moe {

constexpr int kMbRows = 128, kMbCols = 256;
constexpr int kMbThreads = 256;
constexpr int kMbHalfA = kMbRows * 128;
static_assert(kMbRows == kMxBlockTileRows, "tile rows");

struct MbLds {
  uint8_t* b;      // weight tile of the step: 256 rows x 128 bytes
  uint8_t* a;      // token rows, first and second 128 K values of the step (16 KB each)
  uint8_t* bs;     // weight scale bytes [2][256 rows][16]
  uint8_t* as;     // token scale bytes [2][128 rows][16]
  int* tok;        // token (gate_up) or h row (down) of each tile row; -1: none
};

// LDS reads left in flight (lds_read16) until a wait names their registers.
template <int OFF>
__device__ __forceinline__ void mb_read1(uint32_t addr, int& v) {
  asm volatile("ds_read_u8 %0, %1 offset:%2" : "=&v"(v) : "v"(addr), "n"(OFF) : "memory");
}
// A token fragment: 16 rows, 128 K values, and the lane's scale byte.
struct MbFragA {
  v4i lo, hi;
  int s;
};
template <int N>  // all but the newest N LDS reads
__device__ __forceinline__ void mb_wait(MbFragA& f) {
  asm volatile("s_waitcnt lgkmcnt(%3)" : "+v"(f.lo), "+v"(f.hi), "+v"(f.s) : "n"(N) : "memory");
}
template <int N>
__device__ __forceinline__ void mb_wait8(v4i (&b)[8], int (&s)[8]) {
  asm volatile("s_waitcnt lgkmcnt(%16)"
               : "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]), "+v"(b[4]), "+v"(b[5]), "+v"(b[6]),
                 "+v"(b[7]), "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]), "+v"(s[4]), "+v"(s[5]),
                 "+v"(s[6]), "+v"(s[7])
               : "n"(N)
               : "memory");
}

// Weight fragment 4 h + n: column tile n, half h of the step, and its scale byte (ODD: the
// step is the second of its scale group). Column tile n's first tile row, past the
// wave's first: gate_up holds two gate tiles, then the two up tiles of the same columns.
template <int KIND, int ODD>
__device__ __forceinline__ void mb_read_b(uint32_t b_h0, uint32_t b_h1, uint32_t s_addr, v4i (&b)[8],
                                          int (&s)[8]) {
  constexpr int r1 = 16, r2 = KIND == 0 ? 128 : 32, r3 = KIND == 0 ? 144 : 48;
#define MB_B(H, N, R)                                  \
  lds_read16<(R) * 128>(H ? b_h1 : b_h0, b[4 * H + N]); \
  mb_read1<(R) * 16 + 8 * ODD + 4 * H>(s_addr, s[4 * H + N]);
  MB_B(0, 0, 0) MB_B(0, 1, r1) MB_B(0, 2, r2) MB_B(0, 3, r3)
  MB_B(1, 0, 0) MB_B(1, 1, r1) MB_B(1, 2, r2) MB_B(1, 3, r3)
#undef MB_B
}
// Token fragment m (rows 16 m ..) of half H.
template <int H, int ODD>
__device__ __forceinline__ void mb_read_a(uint32_t lo, uint32_t hi, uint32_t s_addr, int m, MbFragA& f) {
#define MB_A(M)                                    \
  case M:                                          \
    lds_read16<kMbHalfA * H + 2048 * M>(lo, f.lo);  \
    lds_read16<kMbHalfA * H + 2048 * M>(hi, f.hi);  \
    mb_read1<8 * ODD + 4 * H + 256 * M>(s_addr, f.s); \
    break;
  switch (m) {
    MB_A(0) MB_A(1) MB_A(2) MB_A(3) MB_A(4) MB_A(5) MB_A(6) MB_A(7)
  }
#undef MB_A
}

// Four scale bytes in one register; mb_mfma's operand select picks byte n.
__device__ __forceinline__ int mb_pack4(const int* s) {
  return s[0] | (s[1] << 8) | (s[2] << 16) | (s[3] << 24);
}
__device__ __forceinline__ v4f mb_mfma(const MbFragA& f, const v4i& b4, const v4f& c, int sb4, int n) {
  const v8i a = {f.lo.x, f.lo.y, f.lo.z, f.lo.w, f.hi.x, f.hi.y, f.hi.z, f.hi.w};
  const v8i b = {b4.x, b4.y, b4.z, b4.w, 0, 0, 0, 0};
  switch (n) {
    case 0: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, kFmtFp8, kFmtFp4, 0, f.s, 0, sb4);
    case 1: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, kFmtFp8, kFmtFp4, 0, f.s, 1, sb4);
    case 2: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, kFmtFp8, kFmtFp4, 0, f.s, 2, sb4);
    default: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, kFmtFp8, kFmtFp4, 0, f.s, 3, sb4);
  }
}

// One work item: rows [slot0, slot0 + nrows) of expert e (hq / y rows from rbase), at most
// 16 MF of them, against column tile nt.
template <int KIND, int MF>
__device__ __forceinline__ void mx_block_item(const MxArgs& p, const MbLds& s, const int e,
                                              const long slot0, const long rbase, const int nrows,
                                              const int nt) {
  constexpr int NA = (MF + 1) / 2;  // token-row loads per wave and half step
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int Kdim = (KIND == 0) ? p.H : p.I;
  const int KS = Kdim / 32;   // scale bytes per row
  const int NS = Kdim / 256;  // steps (even: K % 512 == 0)
  const int wrb = Kdim / 2;   // weight row bytes
  const int rows_w = (KIND == 0) ? 2 * p.I : p.H;
  const long arows = (KIND == 0) ? p.T : p.rows;
  const buf_rsrc_t rw = buf_rsrc(p.w + (size_t)e * rows_w * wrb, (long)rows_w * wrb);
  const buf_rsrc_t rws = buf_rsrc(p.ws + (size_t)e * rows_w * KS, (long)rows_w * KS);
  const buf_rsrc_t ra = buf_rsrc(p.a, arows * Kdim);
  const buf_rsrc_t ras = buf_rsrc(p.as, arows * KS);

  // Tile row -> weight row. Wave w multiplies gate rows 32 w .. 32 w + 31 and the matching
  // up rows (gate_up: one MX block of h), or 64 outputs (down). Row 16 n + j of a wave's
  // part holds output column 2 j + n (gate_up) or 4 j + n (down), so lane j stores
  // consecutive columns.
  auto wrow_of = [&](int row) -> int {
    if (KIND == 0) {
      const int hc = nt * 128 + (row & 96) + 2 * (row & 15) + ((row >> 4) & 1);
      return row < 128 ? hc : p.I + hc;
    }
    return nt * kMbCols + (row & 192) + 4 * (row & 15) + ((row >> 4) & 3);
  };
  // Weight loads: wave w fills tile rows [64 w, +64), load i rows 64 w + 8 i + l / 8,
  // stored chunk l % 8 = logical chunk swz(row, l % 8). Two lane offsets and a uniform
  // step cover the eight.
  uint32_t boff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 64 * wave + 8 * i + (lane >> 3);
    boff[i] = (uint32_t)wrow_of(row) * (uint32_t)wrb + (uint32_t)(swz(row, lane & 7) * 16);
  }
  const uint32_t bsoff = (uint32_t)wrow_of(64 * wave + lane) * (uint32_t)KS;
  auto load_b = [&](int i, int st) {
    const int q = i >> 1, drow = KIND == 0 ? (q & 1) + 32 * (q >> 1) : q;  // rows past boff's
    buf_lds16<true>(rw, boff[i & 1], drow * wrb + st * 128, s.b + (8 * wave + i) * 1024);
  };
  auto load_bs = [&](int grp) { buf_lds16(rws, bsoff, grp * 16, s.bs + (grp & 1) * 4096 + wave * 1024); };
  // token (gate_up) or h row (down) behind a tile row; rows with none read row 0 and are
  // not stored. The token ids are requested before the weight tile (loads return in
  // order, and the token rows' addresses need them).
  auto id_of = [&](int row) -> int {
    return KIND == 0 ? p.tpid[slot0 + min(row, nrows - 1)] : (int)rbase + row;
  };
  auto src_of = [&](int row, int id) -> int {
    return (row < nrows && id >= 0 && (KIND == 1 || id < p.T)) ? id : -1;
  };
  // Token loads: load i of wave w fills rows 8 (w + 4 i) .. + 7 (past the last fragment:
  // the last rows once more, so every wave issues NA loads without a branch, which would
  // split the MFMA sequence); waves 2 and 3 repeat the scale loads of 0 and 1.
  const int srow = 64 * (wave & 1) + lane;
  int areg[NA], aid[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    areg[i] = min(wave + 4 * i, 2 * MF - 1);
    aid[i] = id_of(8 * areg[i] + (lane >> 3));
  }
  const int sid = id_of(srow);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) load_b(i, 0);
  load_bs(0);
  __builtin_amdgcn_sched_barrier(0);
  uint32_t aoff[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int row = 8 * areg[i] + (lane >> 3), src = src_of(row, aid[i]);
    aoff[i] = (uint32_t)(src < 0 ? 0 : src) * (uint32_t)Kdim + (uint32_t)(swz(row, lane & 7) * 16);
  }
  const int ssrc = src_of(srow, sid);
  const uint32_t asoff = (uint32_t)(ssrc < 0 ? 0 : ssrc) * (uint32_t)KS;
  if (KIND == 0 && wave < 2) lds_st32(lds_addr(s.tok) + 4 * srow, ssrc);
  auto load_a = [&](int i, int kb, uint8_t* dst) { buf_lds16(ra, aoff[i], kb * 128, dst + areg[i] * 1024); };
  auto load_as = [&](int grp) {
    buf_lds16(ras, asoff, grp * 16, s.as + (grp & 1) * 2048 + (wave & 1) * 1024);
  };
#pragma unroll
  for (int i = 0; i < NA; ++i) load_a(i, 0, s.a);
  load_as(0);

  v4f acc[MF][4];
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n) acc[m][n] = (v4f){0.f, 0.f, 0.f, 0.f};

  const uint32_t sw = (r16 >> 1) & 7;
  const uint32_t b_base = lds_addr(s.b) + ((KIND == 0 ? 32 : 64) * wave + r16) * 128;
  const uint32_t b_h0 = b_base + ((g ^ sw) << 4), b_h1 = b_base + (((4 + g) ^ sw) << 4);
  const uint32_t a_lo = lds_addr(s.a) + r16 * 128 + ((g ^ sw) << 4);
  const uint32_t a_hi = lds_addr(s.a) + r16 * 128 + (((4 + g) ^ sw) << 4);
  const uint32_t bs_base = lds_addr(s.bs) + ((KIND == 0 ? 32 : 64) * wave + r16) * 16 + g;
  const uint32_t as_base = lds_addr(s.as) + r16 * 16 + g;

  // One step. Its loads, each at the start of a half (so the weight buffer is being
  // refilled for all of the step): in half 0 the step's token half 1, then the next weight
  // tile; in half 1 the next step's token half 0 and, every second step, the next scale
  // group.
  auto step = [&](int st, auto odd_c, auto last_c) {
    constexpr int ODD = decltype(odd_c)::value;     // st & 1: second half of a scale group
    constexpr bool LAST = decltype(last_c)::value;  // last pair of steps
    constexpr bool END = LAST && ODD;               // last step
    constexpr int NB = END ? 0 : 8;                 // weight loads
    wait_vm<0>();   // the weight tile, token half 0 and the scales have landed
    lds_barrier();  // ... for every wave
    const uint32_t bsa = bs_base + (uint32_t)((st >> 1) & 1) * 4096;
    const uint32_t asa = as_base + (uint32_t)((st >> 1) & 1) * 2048;
    v4i b[8];
    int sb[8];
    MbFragA f[3];
    mb_read_b<KIND, ODD>(b_h0, b_h1, bsa, b, sb);
    mb_read_a<0, ODD>(a_lo, a_hi, asa, 0, f[0]);
    mb_wait8<3>(b, sb);
    const int sp[2] = {mb_pack4(sb), mb_pack4(sb + 4)};
    lds_barrier();  // every wave holds its weight fragments (and is done with token half 1)
    auto half = [&](auto h_c) {
      constexpr int Hh = decltype(h_c)::value;
      if (MF > 1) mb_read_a<Hh, ODD>(a_lo, a_hi, asa, 1, f[1]);
      mb_wait<(MF > 1) ? 3 : 0>(f[0]);
#pragma unroll
      for (int m = 0; m < MF; ++m) {
        if (m + 2 < MF) mb_read_a<Hh, ODD>(a_lo, a_hi, asa, m + 2, f[(m + 2) % 3]);
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          __builtin_amdgcn_sched_barrier(0);
          acc[m][n] = mb_mfma(f[m % 3], b[4 * Hh + n], acc[m][n], sp[Hh], n);
          __builtin_amdgcn_sched_barrier(0);
          if (m == 0 && n == 0) {
            if (Hh == 0) {
#pragma unroll
              for (int i = 0; i < NA; ++i) load_a(i, 2 * st + 1, s.a + kMbHalfA);
#pragma unroll
              for (int i = 0; i < NB; ++i) load_b(i, st + 1);
            } else if (!END) {
#pragma unroll
              for (int i = 0; i < NA; ++i) load_a(i, 2 * st + 2, s.a);
              if (!ODD && !LAST) {
                load_bs((st >> 1) + 1);
                load_as((st >> 1) + 1);
              }
            }
          }
        }
        acc_pin(acc[m > 0 ? m - 1 : MF - 1]);
        if (m + 1 < MF) {
          if (m + 2 < MF)
            mb_wait<3>(f[(m + 1) % 3]);
          else
            mb_wait<0>(f[(m + 1) % 3]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    half(std::integral_constant<int, 0>{});
    wait_vm<NB>();   // token half 1 has landed
    lds_barrier();   // ... for every wave; token half 0 is read
    mb_read_a<1, ODD>(a_lo, a_hi, asa, 0, f[0]);
    half(std::integral_constant<int, 1>{});
  };
  const std::integral_constant<int, 0> even{};
  const std::integral_constant<int, 1> odd{};
  for (int st = 0; st < NS - 2; st += 2) {
    step(st, even, std::false_type{});
    step(st + 1, odd, std::false_type{});
  }
  step(NS - 2, even, std::true_type{});
  step(NS - 1, odd, std::true_type{});

  // Epilogue. Lane l, register i of acc[m][n] holds row 16 m + 4 (l / 16) + i and output
  // column 2 (l % 16) + n (gate_up, n < 2; n + 2: the up value) or 4 (l % 16) + n (down) of
  // the wave's.
  const float* bias = p.bias == nullptr ? nullptr : p.bias + (size_t)e * rows_w;
  // (lane indices taken anew: the store addresses are not held through the K loop)
  int el = lane;
  asm volatile("" : "+v"(el));
  const int eg = el >> 4, e16 = el & 15;
  if (KIND == 0) {
    const int hc = nt * 128 + 32 * wave + 2 * e16;
    float bg[2] = {0.f, 0.f}, bu[2] = {0.f, 0.f};
    if (bias != nullptr) {
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        bg[n] = bias[hc + n];
        bu[n] = bias[p.I + hc + n];
      }
    }
    const int GI = p.I / 32;
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float h[2], mx = 0.f;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          const float gt = fminf(fmaxf(acc[m][n][i] + bg[n], p.gate_lo), p.gate_hi);
          const float up = fminf(fmaxf(acc[m][n + 2][i] + bu[n], p.up_lo), p.up_hi);
          h[n] = mx_act(gt, p.act) * up;
          mx = fmaxf(mx, fabsf(h[n]));
        }
        mx = group16_max_f32(mx);  // 16 lanes hold the 32 columns of one MX block
        const int ex = mx_exponent(mx);
        const int row = 16 * m + 4 * eg + i;
        const uint32_t c2 = mx_e4m3x2(h[0], h[1], mx_inv_scale(ex));
        if (row < nrows && s.tok[row] >= 0) {
          *(uint16_t*)(p.hq + (size_t)(rbase + row) * p.I + hc) = (uint16_t)c2;
          if (e16 == 0) p.hs[(size_t)(rbase + row) * GI + (hc >> 5)] = (uint8_t)(ex + 127);
        }
      }
  } else {
    const int oc = nt * kMbCols + 64 * wave + 4 * e16;
    float bo[4] = {0.f, 0.f, 0.f, 0.f};
    if (bias != nullptr) {
#pragma unroll
      for (int n = 0; n < 4; ++n) bo[n] = bias[oc + n];
    }
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 16 * m + 4 * eg + i;
        uint2 o;
        o.x = bf16x2(acc[m][0][i] + bo[0], acc[m][1][i] + bo[1]);
        o.y = bf16x2(acc[m][2][i] + bo[2], acc[m][3][i] + bo[3]);
        if (row < nrows) *(uint2*)(p.y + (size_t)(rbase + row) * p.H + oc) = o;
      }
  }
}

// Block tiles (p.seg set) or row tiles.
template <int KIND>
__global__ __launch_bounds__(kMbThreads, 2) void expert_gemm_mx_block_kernel(MxArgs p) {
  __shared__ __attribute__((aligned(1024))) uint8_t sB[kMbCols * 128];
  __shared__ __attribute__((aligned(1024))) uint8_t sA[2 * kMbHalfA];
  __shared__ __attribute__((aligned(1024))) uint8_t sBS[2 * kMbCols * 16];
  __shared__ __attribute__((aligned(1024))) uint8_t sAS[2 * kMbRows * 16];
  __shared__ int sTok[kMbRows];
  const MbLds s{sB, sA, sBS, sAS, sTok};
  const int NT = (KIND == 0) ? p.I / 128 : p.H / kMbCols;
  int tile, nt;
  if (p.seg != nullptr) {
    // XCD-aware item index, as in the fp8 block kernels: XCD x takes the items of tiles
    // [cut[x], cut[x + 1]) of the list's header, expert by expert and column tile by
    // column tile, so the row tiles of an expert share each weight tile in one L2.
    const int x = blockIdx.x & 7;
    const int L = p.num_tiles[1 + x] * NT + (int)(blockIdx.x >> 3);
    if (L >= p.num_tiles[2 + x] * NT) return;
    const int2 sg = p.seg[L / NT];
    const int r0 = L - NT * sg.x;
    nt = r0 / sg.y;
    tile = sg.x + (r0 - nt * sg.y);
  } else {
    tile = blockIdx.x / NT;
    nt = blockIdx.x - tile * NT;
  }
  if (tile >= p.num_tiles[0]) return;  // past the list, or a truncated one
  // (wave-uniform, so the operand bases stay in scalar registers)
  const int4 tv = p.tiles[tile];
  const int4 td = make_int4(__builtin_amdgcn_readfirstlane(tv.x), __builtin_amdgcn_readfirstlane(tv.y),
                            __builtin_amdgcn_readfirstlane(tv.z), __builtin_amdgcn_readfirstlane(tv.w));
  const int e = td.x, nrows = td.z;
  if (e < 0 || e >= p.E || nrows <= 0 || nrows > kMbRows) return;
  switch ((nrows + 15) / 16) {
    case 1: return mx_block_item<KIND, 1>(p, s, e, td.y, td.w, nrows, nt);
    case 2: return mx_block_item<KIND, 2>(p, s, e, td.y, td.w, nrows, nt);
    case 3: return mx_block_item<KIND, 3>(p, s, e, td.y, td.w, nrows, nt);
    case 4: return mx_block_item<KIND, 4>(p, s, e, td.y, td.w, nrows, nt);
    case 5: return mx_block_item<KIND, 5>(p, s, e, td.y, td.w, nrows, nt);
    case 6: return mx_block_item<KIND, 6>(p, s, e, td.y, td.w, nrows, nt);
    case 7: return mx_block_item<KIND, 7>(p, s, e, td.y, td.w, nrows, nt);
    default: return mx_block_item<KIND, 8>(p, s, e, td.y, td.w, nrows, nt);
  }
}

bool mx_block_fits(int kind, const MxArgs& a) {
  auto al = [](const void* q, uintptr_t n) { return ((uintptr_t)q & (n - 1)) == 0; };
  const unsigned long lim = 1UL << 32;
  return a.nsh == 0 && a.H % 512 == 0 && a.I % 512 == 0 && al(a.a, 16) && al(a.as, 16) && al(a.w, 16) &&
         al(a.ws, 16) && al(a.hq, 2) && al(a.y, 8) &&
         (unsigned long)(kind == 0 ? a.T : a.rows) * (unsigned long)(kind == 0 ? a.H : a.I) < lim &&
         (unsigned long)a.I * a.H < lim && a.rows < (1L << 31);
}

void launch_mx_block(int kind, const MxArgs& a, int max_tiles, hipStream_t st) {
  const long NT = (kind == 0) ? a.I / 128 : a.H / kMbCols;
  // block tiles: each XCD's share of them
  const long items = (a.seg != nullptr ? 8L * block_tiles_cap(max_tiles) : (long)max_tiles) * NT;
  if (kind == 0)
    hipLaunchKernelGGL(expert_gemm_mx_block_kernel<0>, dim3((unsigned)items), dim3(kMbThreads), 0, st, a);
  else
    hipLaunchKernelGGL(expert_gemm_mx_block_kernel<1>, dim3((unsigned)items), dim3(kMbThreads), 0, st, a);
}

}  // namespace moe

int moe::mx_block_max_tiles(int T, int K, int E) {
  const long rows = (long)T * std::min(K, E);
  return (int)(rows / kMxBlockTileRows + std::min<long>(E, rows));
}
