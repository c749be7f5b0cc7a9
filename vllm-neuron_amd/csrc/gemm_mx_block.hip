// Prefill-sized MXFP4 expert GEMMs (GPT-OSS), for the layer above 32 routed rows per
// expert. Same products, epilogue arithmetic and K order as the row-tile kernel
// (gemm_mx.hip), on tiles tall enough that the matrix cores, not the weight stream of
// one 64-row tile, set the time.
//
//  * A workgroup of 4 waves computes up to 128 rows x 256 weight rows (gate_up: 128
//    gate rows + the matching 128 up rows; down: 256 outputs). Wave (wm, wn) owns 16 MF
//    rows (MF = ceil(tile rows / 32)) and 128 columns: MF x 8 tiles of
//    v_mfma_scale_f32_16x16x128_f8f6f4, whose E8M0 operands apply every block scale.
//  * 76.5 KB of LDS, so two workgroups share a CU (two waves per SIMD). They meet no
//    common barrier: one's fragment reads, waits, prologue and epilogue run under the
//    other's MFMAs. One workgroup of eight waves reads all its fragments at the same
//    moment instead and leaves the matrix cores idle meanwhile.
//  * A step is 256 K values: 128 bytes of every weight row (whole cache lines) and two
//    128-byte pieces of every token row, by direct-to-LDS loads. The weight tile has one
//    32 KB buffer: half 1's fragments move to registers during half 0's last MFMAs, so
//    the buffer is refilled at mid-step; each token half has its own 16 KB buffer,
//    refilled as soon as its fragments are read. Every wait is for all loads of the
//    previous half step.
//  * The scale bytes of 512 K values (16 per row) arrive with one 16-byte load per row
//    every second step.
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

struct MxBlkArgs {
  MxArgs m;
  const int2* seg;  // {first tile of the expert, tiles of the expert}
};

struct MbLds {
  uint8_t* b;      // weight tile of the step: 256 rows x 128 bytes
  uint8_t* a;      // token rows, first and second 128 K values of the step (16 KB each)
  uint8_t* bs;     // weight scale bytes [2][256 rows][16]
  uint8_t* as;     // token scale bytes [2][128 rows][16]
  int* tok;        // token (gate_up) or h row (down) of each tile row; -1: none
};

// LDS reads left in flight until mb_wait names their registers (LDS reads complete in
// order). In asm, because the compiler would wait for every direct-to-LDS load in flight
// before a plain read.
__device__ __forceinline__ void lds_st32(uint32_t addr, int v) {
  asm volatile("ds_write_b32 %0, %1" : : "v"(addr), "v"(v) : "memory");
}
template <int OFF>
__device__ __forceinline__ void mb_read16(uint32_t addr, v4i& v) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(v) : "v"(addr), "n"(OFF) : "memory");
}
template <int OFF>
__device__ __forceinline__ void mb_read1(uint32_t addr, int& v) {
  asm volatile("ds_read_u8 %0, %1 offset:%2" : "=&v"(v) : "v"(addr), "n"(OFF) : "memory");
}
__device__ __forceinline__ void mb_wait(v4i& a, v4i& b, int& s) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a), "+v"(b), "+v"(s) : : "memory");
}
__device__ __forceinline__ void mb_wait8(v4i (&b)[8], int (&s)[8]) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]), "+v"(b[4]), "+v"(b[5]), "+v"(b[6]),
                 "+v"(b[7]), "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]), "+v"(s[4]), "+v"(s[5]),
                 "+v"(s[6]), "+v"(s[7])
               :
               : "memory");
}

// Keeps eight accumulators' MFMAs before this point (nothing is read): the compiler
// otherwise delays MFMAs past the reads of the next fragments, whose registers then pile
// up. Placed one row group behind, so no MFMA result is still on its way.
__device__ __forceinline__ void mb_pin(v4f (&c)[8]) {
  asm volatile("" : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[3]), "+v"(c[4]), "+v"(c[5]), "+v"(c[6]), "+v"(c[7]));
}

// Weight fragment n of half H of a step (and its scale byte; ODD: the step is the second
// of its scale group): the tile row of its first row is
// kRow[n] past the wave's first row.
template <int KIND>
struct MbRow {
  static constexpr int at(int n) { return KIND == 0 ? (n < 4 ? 16 * n : 128 + 16 * (n - 4)) : 16 * n; }
};
template <int KIND, int H, int ODD>
__device__ __forceinline__ void mb_read_b(uint32_t b_addr, uint32_t s_addr, int n, v4i& b, int& s) {
#define MB_B(N)                                                 \
  case N:                                                       \
    mb_read16<MbRow<KIND>::at(N) * 128>(b_addr, b);             \
    mb_read1<MbRow<KIND>::at(N) * 16 + 8 * ODD + 4 * H>(s_addr, s);               \
    break;
  switch (n) {
    MB_B(0) MB_B(1) MB_B(2) MB_B(3) MB_B(4) MB_B(5) MB_B(6)
    default:
      mb_read16<MbRow<KIND>::at(7) * 128>(b_addr, b);
      mb_read1<MbRow<KIND>::at(7) * 16 + 8 * ODD + 4 * H>(s_addr, s);
      break;
  }
#undef MB_B
}
// Token fragment m of half H (16 rows at 16 m of the wave's row group) and its scale byte.
template <int H, int ODD>
__device__ __forceinline__ void mb_read_a(uint32_t lo, uint32_t hi, uint32_t s_addr, int m, v4i& alo,
                                          v4i& ahi, int& s) {
#define MB_A(M)                                 \
  mb_read16<kMbHalfA * H + 2048 * M>(lo, alo);  \
  mb_read16<kMbHalfA * H + 2048 * M>(hi, ahi);  \
  mb_read1<8 * ODD + 4 * H + 256 * M>(s_addr, s);
  switch (m) {
    case 0: MB_A(0) break;
    case 1: MB_A(1) break;
    case 2: MB_A(2) break;
    default: MB_A(3) break;
  }
#undef MB_A
}

// Four scale bytes in one register; mb_mfma's operand select picks byte n % 4.
__device__ __forceinline__ int mb_pack4(const int* s) {
  return s[0] | (s[1] << 8) | (s[2] << 16) | (s[3] << 24);
}
__device__ __forceinline__ v4f mb_mfma(const v8i& a, const v4i& b4, const v4f& c, int sa, int sb4, int n) {
  const v8i b = {b4.x, b4.y, b4.z, b4.w, 0, 0, 0, 0};
  switch (n & 3) {
    case 0: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, kFmtFp8, kFmtFp4, 0, sa, 0, sb4);
    case 1: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, kFmtFp8, kFmtFp4, 0, sa, 1, sb4);
    case 2: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, kFmtFp8, kFmtFp4, 0, sa, 2, sb4);
    default: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, kFmtFp8, kFmtFp4, 0, sa, 3, sb4);
  }
}

// One work item: rows [slot0, slot0 + nrows) of expert e (hq / y rows from rbase)
// against column tile nt.
template <int KIND, int MF>
__device__ __forceinline__ void mx_block_item(const MxArgs& p, const MbLds& s, const int e,
                                              const long slot0, const long rbase, const int nrows,
                                              const int nt) {
  constexpr int RG = 16 * MF;  // rows per row group
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
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

  // Tile row -> weight row: column tile n of a wave reads tile rows 16 n + j, and they
  // hold output columns 4 j + n (gate_up, per 64-column wave half) or 8 j + n (down, per
  // 128-column half), so lane j stores consecutive output columns.
  auto wrow_of = [&](int row) -> int {
    if (KIND == 0) {
      const int r = row & 127;
      const int hc = (r & 64) + 4 * (r & 15) + ((r >> 4) & 3);
      return (row < 128) ? nt * 128 + hc : p.I + nt * 128 + hc;
    }
    return nt * kMbCols + (row & 128) + 8 * (row & 15) + ((row >> 4) & 7);
  };
  // Weight loads: wave w fills tile rows [64 w, +64), load i rows 64 w + 8 i + l / 8,
  // stored chunk l % 8 = logical chunk swz(row, l % 8). Rows 8 i + c and 8 (i + 2) + c
  // are one weight row apart, so two lane offsets and a uniform step cover the eight.
  uint32_t boff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 64 * wave + 8 * i + (lane >> 3);
    boff[i] = (uint32_t)wrow_of(row) * (uint32_t)wrb + (uint32_t)(swz(row, lane & 7) * 16);
  }
  const uint32_t bsoff = (uint32_t)wrow_of(64 * wave + lane) * (uint32_t)KS;
  auto load_b = [&](int i, int st) {
    buf_lds16(rw, boff[i & 1], (i >> 1) * wrb + st * 128, s.b + (8 * wave + i) * 1024);
  };
  auto load_bs = [&](int grp) {
    buf_lds16(rws, bsoff, grp * 16, s.bs + (grp & 1) * 4096 + wave * 1024);
  };
  // token (gate_up) or h row (down) behind a tile row; rows with none read row 0 and are
  // not stored. The token ids are requested before the weight tile (loads return in
  // order, and the token rows' addresses need them).
  auto id_of = [&](int row) -> int {
    return KIND == 0 ? p.tpid[slot0 + min(row, nrows - 1)] : (int)rbase + row;
  };
  auto src_of = [&](int row, int id) -> int {
    return (row < nrows && id >= 0 && (KIND == 1 || id < p.T)) ? id : -1;
  };
  const int srow = 64 * (wave & 1) + lane;
  int arow[MF], aid[MF];
#pragma unroll
  for (int i = 0; i < MF; ++i) {
    arow[i] = 8 * (MF * wave + i) + (lane >> 3);
    aid[i] = id_of(arow[i]);
  }
  const int sid = id_of(srow);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) load_b(i, 0);
  load_bs(0);
  __builtin_amdgcn_sched_barrier(0);
  uint32_t aoff[MF];
#pragma unroll
  for (int i = 0; i < MF; ++i) {
    const int src = src_of(arow[i], aid[i]);
    aoff[i] = (uint32_t)(src < 0 ? 0 : src) * (uint32_t)Kdim + (uint32_t)(swz(arow[i], lane & 7) * 16);
  }
  const int ssrc = src_of(srow, sid);
  const uint32_t asoff = (uint32_t)(ssrc < 0 ? 0 : ssrc) * (uint32_t)KS;
  if (KIND == 0 && wave < 2) lds_st32(lds_addr(s.tok) + 4 * srow, ssrc);
  auto load_a = [&](int i, int kb, uint8_t* dst) {
    buf_lds16(ra, aoff[i], kb * 128, dst + (MF * wave + i) * 1024);
  };
  auto load_as = [&](int grp) {
    // waves 2 and 3 repeat the loads of 0 and 1: a branch would split the MFMA sequence
    buf_lds16(ras, asoff, grp * 16, s.as + (grp & 1) * 2048 + (wave & 1) * 1024);
  };
#pragma unroll
  for (int i = 0; i < MF; ++i) load_a(i, 0, s.a);
  load_as(0);

  v4f acc[MF][8];
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int n = 0; n < 8; ++n) acc[m][n] = (v4f){0.f, 0.f, 0.f, 0.f};

  const uint32_t sw = (r16 >> 1) & 7;
  const uint32_t b_base = lds_addr(s.b) + ((KIND == 0 ? 64 : 128) * wn + r16) * 128;
  const uint32_t b_h0 = b_base + ((g ^ sw) << 4), b_h1 = b_base + (((4 + g) ^ sw) << 4);
  const uint32_t f_lo = (RG * wm + r16) * 128 + ((g ^ sw) << 4);
  const uint32_t f_hi = (RG * wm + r16) * 128 + (((4 + g) ^ sw) << 4);
  const uint32_t a_lo = lds_addr(s.a) + f_lo, a_hi = lds_addr(s.a) + f_hi;
  const uint32_t bs_base = lds_addr(s.bs) + ((KIND == 0 ? 64 : 128) * wn + r16) * 16 + g;
  const uint32_t as_base = lds_addr(s.as) + (RG * wm + r16) * 16 + g;

  // One step. Its token half 1 and the next step's weight tile, token half 0 and scales
  // are loaded meanwhile, spread among the MFMAs.
  auto step = [&](int st, auto odd_c, auto last_c) {
    constexpr int ODD = decltype(odd_c)::value;     // st & 1: second half of a scale group
    constexpr bool LAST = decltype(last_c)::value;  // last pair of steps
    wait_vm<0>();   // the weight tile, token half 0 and the scales have landed
    lds_barrier();  // ... for every wave, and the last step's token half 1 is read
    const uint32_t bsa = bs_base + (uint32_t)((st >> 1) & 1) * 4096;
    const uint32_t asa = as_base + (uint32_t)((st >> 1) & 1) * 2048;
    v4i b[8], bn[8];
    int sb[8], sbn[8];
#pragma unroll
    for (int n = 0; n < 8; ++n) mb_read_b<KIND, 0, ODD>(b_h0, bsa, n, b[n], sb[n]);
    v4i alo, ahi, nlo, nhi;
    int sa, nsa;
    mb_read_a<0, ODD>(a_lo, a_hi, asa, 0, alo, ahi, sa);
    mb_wait8(b, sb);
    int sp[2] = {mb_pack4(sb), mb_pack4(sb + 4)};
    mb_wait(alo, ahi, sa);
    __builtin_amdgcn_sched_barrier(0);
    // half 0
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      if (m + 1 < MF) mb_read_a<0, ODD>(a_lo, a_hi, asa, m + 1, nlo, nhi, nsa);
      const v8i a = (v8i){alo.x, alo.y, alo.z, alo.w, ahi.x, ahi.y, ahi.z, ahi.w};
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        __builtin_amdgcn_sched_barrier(0);
        acc[m][n] = mb_mfma(a, b[n], acc[m][n], sa, sp[n >> 2], n);
        __builtin_amdgcn_sched_barrier(0);
        if (m == MF - 1) mb_read_b<KIND, 1, ODD>(b_h1, bsa, n, bn[n], sbn[n]);
        // token half 1 (MF loads), then, every second step, the next scale group
        if (m == 0 && n < MF) load_a(n, 2 * st + 1, s.a + kMbHalfA);
        if (m == 0 && n == 4 && !LAST && ODD == 0) {
          load_bs((st >> 1) + 1);
          load_as((st >> 1) + 1);
        }
      }
      mb_pin(acc[m > 0 ? m - 1 : MF - 1]);
      if (m + 1 < MF) {
        mb_wait(nlo, nhi, nsa);
        alo = nlo;
        ahi = nhi;
        sa = nsa;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    mb_wait8(bn, sbn);
    sp[0] = mb_pack4(sbn);
    sp[1] = mb_pack4(sbn + 4);
    wait_vm<0>();   // token half 1 has landed
    lds_barrier();  // ... for every wave; the weight tile and token half 0 are read
    mb_read_a<1, ODD>(a_lo, a_hi, asa, 0, alo, ahi, sa);
    mb_wait(alo, ahi, sa);
    __builtin_amdgcn_sched_barrier(0);
    // half 1
    constexpr int kLoads = 8 + MF, kPos = 8 * MF;
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      if (m + 1 < MF) mb_read_a<1, ODD>(a_lo, a_hi, asa, m + 1, nlo, nhi, nsa);
      const v8i a = (v8i){alo.x, alo.y, alo.z, alo.w, ahi.x, ahi.y, ahi.z, ahi.w};
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        __builtin_amdgcn_sched_barrier(0);
        acc[m][n] = mb_mfma(a, bn[n], acc[m][n], sa, sp[n >> 2], n);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!(LAST && ODD)) {
          // load j at MFMA floor(j kPos / kLoads): the weight tile, then token half 0
          const int pos = 8 * m + n;
#pragma unroll
          for (int j = 0; j < kLoads; ++j) {
            if (j * kPos / kLoads == pos) {
              if (j < 8)
                load_b(j, st + 1);
              else
                load_a(j - 8, 2 * st + 2, s.a);
            }
          }
        }
      }
      mb_pin(acc[m > 0 ? m - 1 : MF - 1]);
      if (m + 1 < MF) {
        mb_wait(nlo, nhi, nsa);
        alo = nlo;
        ahi = nhi;
        sa = nsa;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  const std::integral_constant<int, 0> even{};
  const std::integral_constant<int, 1> odd{};
  for (int st = 0; st < NS - 2; st += 2) {
    step(st, even, std::false_type{});
    step(st + 1, odd, std::false_type{});
  }
  step(NS - 2, even, std::true_type{});
  step(NS - 1, odd, std::true_type{});

  // Epilogue. Lane l, register i of acc[m][n] holds row RG wm + 16 m + 4 (l / 16) + i and
  // output column 4 (l % 16) + n (gate_up; n + 4: the up value) or 8 (l % 16) + n (down).
  const float* bias = p.bias == nullptr ? nullptr : p.bias + (size_t)e * rows_w;
  // (lane indices taken anew: the store addresses are not held through the K loop)
  int el = lane;
  asm volatile("" : "+v"(el));
  const int eg = el >> 4, e16 = el & 15;
  if (KIND == 0) {
    const int hc = nt * 128 + 64 * wn + 4 * e16;
    float bg[4] = {0.f, 0.f, 0.f, 0.f}, bu[4] = {0.f, 0.f, 0.f, 0.f};
    if (bias != nullptr) {
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        bg[n] = bias[hc + n];
        bu[n] = bias[p.I + hc + n];
      }
    }
    const int GI = p.I / 32;
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float h[4], mx = 0.f;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          const float gt = fminf(fmaxf(acc[m][n][i] + bg[n], p.gate_lo), p.gate_hi);
          const float up = fminf(fmaxf(acc[m][n + 4][i] + bu[n], p.up_lo), p.up_hi);
          h[n] = mx_act(gt, p.act) * up;
          mx = fmaxf(mx, fabsf(h[n]));
        }
        // eight lanes hold the 32 columns of one MX block
#pragma unroll
        for (int o = 4; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
        const int ex = mx_exponent(mx);
        const float f = mx_inv_scale(ex);
        const int row = RG * wm + 16 * m + 4 * eg + i;
        const uint32_t c4 = mx_e4m3x2(h[0], h[1], f) | (mx_e4m3x2(h[2], h[3], f) << 16);
        if (row < nrows && s.tok[row] >= 0) {
          *(uint32_t*)(p.hq + (size_t)(rbase + row) * p.I + hc) = c4;
          if ((e16 & 7) == 0) p.hs[(size_t)(rbase + row) * GI + (hc >> 5)] = (uint8_t)(ex + 127);
        }
      }
  } else {
    const int oc = nt * kMbCols + 128 * wn + 8 * e16;
    float bo[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (bias != nullptr) {
#pragma unroll
      for (int n = 0; n < 8; ++n) bo[n] = bias[oc + n];
    }
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = RG * wm + 16 * m + 4 * eg + i;
        int4 o;
        o.x = (int)bf16x2(acc[m][0][i] + bo[0], acc[m][1][i] + bo[1]);
        o.y = (int)bf16x2(acc[m][2][i] + bo[2], acc[m][3][i] + bo[3]);
        o.z = (int)bf16x2(acc[m][4][i] + bo[4], acc[m][5][i] + bo[5]);
        o.w = (int)bf16x2(acc[m][6][i] + bo[6], acc[m][7][i] + bo[7]);
        if (row < nrows) *(int4*)(p.y + (size_t)(rbase + row) * p.H + oc) = o;
      }
  }
}

template <int KIND>
__global__ __launch_bounds__(kMbThreads, 2) void expert_gemm_mx_block_kernel(MxBlkArgs a) {
  __shared__ __attribute__((aligned(1024))) uint8_t sB[kMbCols * 128];
  __shared__ __attribute__((aligned(1024))) uint8_t sA[2 * kMbHalfA];
  __shared__ __attribute__((aligned(1024))) uint8_t sBS[2 * kMbCols * 16];
  __shared__ __attribute__((aligned(1024))) uint8_t sAS[2 * kMbRows * 16];
  __shared__ int sTok[kMbRows];
  const MbLds s{sB, sA, sBS, sAS, sTok};
  const MxArgs& p = a.m;
  // XCD-aware item index, as in the fp8 block kernels: XCD x takes the items of tiles
  // [cut[x], cut[x + 1]) of the list's header, expert by expert and column tile by
  // column tile, so the row tiles of an expert share each weight tile in one L2.
  const int NT = (KIND == 0) ? p.I / 128 : p.H / kMbCols;
  const int x = blockIdx.x & 7;
  const int L = p.num_tiles[1 + x] * NT + (int)(blockIdx.x >> 3);
  if (L >= p.num_tiles[2 + x] * NT) return;
  const int2 sg = a.seg[L / NT];
  const int r0 = L - NT * sg.x;
  const int nt = r0 / sg.y;
  const int tile = sg.x + (r0 - nt * sg.y);
  if (tile >= p.num_tiles[0]) return;  // truncated tile list
  // (wave-uniform, so the operand bases stay in scalar registers)
  const int4 tv = p.tiles[tile];
  const int4 td = make_int4(__builtin_amdgcn_readfirstlane(tv.x), __builtin_amdgcn_readfirstlane(tv.y),
                            __builtin_amdgcn_readfirstlane(tv.z), __builtin_amdgcn_readfirstlane(tv.w));
  const int e = td.x, nrows = td.z;
  if (e < 0 || e >= p.E || nrows <= 0 || nrows > kMbRows) return;
  if (nrows > 96)
    mx_block_item<KIND, 4>(p, s, e, td.y, td.w, nrows, nt);
  else if (nrows > 64)
    mx_block_item<KIND, 3>(p, s, e, td.y, td.w, nrows, nt);
  else if (nrows > 32)
    mx_block_item<KIND, 2>(p, s, e, td.y, td.w, nrows, nt);
  else
    mx_block_item<KIND, 1>(p, s, e, td.y, td.w, nrows, nt);
}

template <int KIND>
static void launch_mx_block(const MxBlkArgs& a, int max_tiles, hipStream_t st) {
  const int NT = (KIND == 0) ? a.m.I / 128 : a.m.H / kMbCols;
  const long items = 8L * block_tiles_cap(max_tiles) * NT;  // each XCD's share of the tiles
  hipLaunchKernelGGL(expert_gemm_mx_block_kernel<KIND>, dim3((unsigned)items), dim3(kMbThreads), 0, st, a);
}

}  // namespace moe

using namespace moe;

int moe::mx_block_max_tiles(int T, int K, int E) {
  const long rows = (long)T * std::min(K, E);
  return (int)(rows / kMxBlockTileRows + std::min<long>(E, rows));
}

bool moe::mx_block_ok(int T, int H, int I, int E, int K, int wfmt, const void* w13,
                      const void* w13_scale, const void* w2, const void* w2_scale) {
  const unsigned long rows = (unsigned long)T * std::min(K, E);
  auto a16 = [](const void* q) { return ((uintptr_t)q & 15) == 0; };
  return wfmt == MOE_MX_FP4 && H % 512 == 0 && I % 512 == 0 && a16(w13) && a16(w13_scale) && a16(w2) &&
         a16(w2_scale) && (unsigned long)T * H < (1UL << 32) && rows * I < (1UL << 32) &&
         (unsigned long)I * H < (1UL << 32);
}

int moe::layer_gate_up_mx_block(const uint8_t* xq, const uint8_t* xs, int T, int H, int I, int E,
                                const uint8_t* w13, const uint8_t* w13_scale, const float* b13,
                                const int32_t* token_position_to_id, const int32_t* tiles,
                                const int32_t* seg, const int32_t* num_tiles, int max_tiles, int act,
                                float gate_lo, float gate_hi, float up_lo, float up_hi, uint8_t* hq,
                                uint8_t* hs, void* stream) {
  MOE_API_BEGIN("moe_expert_gate_up_mx");
  MOE_CHECK_ARG(xq && xs && w13 && w13_scale && token_position_to_id && tiles && seg && num_tiles && hq && hs,
                "null pointer argument");
  MOE_CHECK_ARG(act == MOE_ACT_SILU || act == MOE_ACT_SWISH, "act must be MOE_ACT_SILU or MOE_ACT_SWISH");
  auto lim = [](float v, float dflt) { return v != v ? dflt : v; };
  MxBlkArgs a{};
  a.m.a = xq;
  a.m.as = xs;
  a.m.w = w13;
  a.m.ws = w13_scale;
  a.m.bias = b13;
  a.m.tpid = token_position_to_id;
  a.m.tiles = (const int4*)tiles;
  a.m.num_tiles = num_tiles;
  a.m.hq = hq;
  a.m.hs = hs;
  a.m.T = T;
  a.m.H = H;
  a.m.I = I;
  a.m.E = E;
  a.m.act = act;
  a.m.gate_lo = lim(gate_lo, -__builtin_inff());
  a.m.gate_hi = lim(gate_hi, __builtin_inff());
  a.m.up_lo = lim(up_lo, -__builtin_inff());
  a.m.up_hi = lim(up_hi, __builtin_inff());
  a.seg = (const int2*)seg;
  launch_mx_block<0>(a, max_tiles, (hipStream_t)stream);
  MOE_API_END();
}

int moe::layer_down_mx_block(const uint8_t* hq, const uint8_t* hs, int T, int H, int I, int E,
                             const uint8_t* w2, const uint8_t* w2_scale, const float* b2,
                             const int32_t* tiles, const int32_t* seg, const int32_t* num_tiles,
                             int max_tiles, long rows, void* y_bf16, void* stream) {
  MOE_API_BEGIN("moe_expert_down_mx");
  MOE_CHECK_ARG(hq && hs && w2 && w2_scale && tiles && seg && num_tiles && y_bf16, "null pointer argument");
  MxBlkArgs a{};
  a.m.a = hq;
  a.m.as = hs;
  a.m.w = w2;
  a.m.ws = w2_scale;
  a.m.bias = b2;
  a.m.tiles = (const int4*)tiles;
  a.m.num_tiles = num_tiles;
  a.m.y = (uint16_t*)y_bf16;
  a.m.rows = rows;
  a.m.T = T;
  a.m.H = H;
  a.m.I = I;
  a.m.E = E;
  a.seg = (const int2*)seg;
  launch_mx_block<1>(a, max_tiles, (hipStream_t)stream);
  MOE_API_END();
}
