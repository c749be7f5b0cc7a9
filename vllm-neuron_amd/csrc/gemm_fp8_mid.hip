// FP8-blockwise expert GEMMs on row tiles of up to 64 rows and block tiles of up to 128, between
// one-token decode and prefill: the weight stream sets the time.
//
// One 16x16x128 MFMA per 128-K scale block, in the arithmetic of the kernels it stands in for,
// so h and y are the same bits: on row tiles acc += part * (s_a[row, k] * s_w[k])
// (gemm_fp8.hip), on block tiles acc = acc * (s_{k-1} / s_k) + part, then acc * s_last, with
// s_k = s_a[row, k] * s_w[k] (gemm_fp8_block.hip).
//
//  * a workgroup of 4 waves computes up to 64 rows x 256 weight rows (gate_up: 128 gate
//    rows + the matching 128 up rows; down: 256 outputs), wave w all rows against 64 of
//    them. 52 KB of LDS and at most 168 registers, so three workgroups share a CU: while one
//    waits, reads its fragments, starts or stores, the others stream and multiply. The ring
//    kernels' one workgroup per CU (one wave per SIMD) leaves its fragment reads, scale
//    multiplies and epilogues in the open, which shows from a few rows per expert on;
//  * the weight tile of a K step (128 values, one cache line per row) has one 32 KB buffer.
//    A wave moves its fragments to registers at the start of the step and the next
//    tile is on its way for the rest of it. The token rows have two 8 KB buffers;
//  * the weights are the MFMA's row operand, so a lane's accumulators belong to one token:
//    its scale (or scale ratio) is one value per fragment, and 8 (gate_up) or 16 (down)
//    consecutive output columns are the lane's own stores;
//  * activation scales of four K blocks per row come with one 16-byte load every fourth
//    step, weight block scales once per tile.
//
//  * tiles of up to 128 rows (block tiles only) keep the same step with 72 KB of LDS and 256
//    registers, two workgroups per CU, and read the token fragments two ahead. An expert
//    of 65 to 128 rows then reads its weights once. Layer, block -> 128-row kernels: Kimi-K2
//    2048 tokens (43 rows per expert) 3214 -> 3129 us, GLM-4.5 1500 tokens (75) 920 -> 863 us.
//    Tried on them: weight fragments straight to registers, without LDS (16 rows x 64 bytes a
//    load: 3883 and 1211 us), the weight loads spread over the step (3210, 899), wave priority
//    for the MFMAs (3134, 865).
//
// Measured where the rules of its use stand (gemm_fp8.hip launch_gemm, kMidTallMaxRows): DeepSeek-V3
// at 600 tokens 11.3 GB of weights in a layer of 1841 us, 6.1 TB/s (ring kernels 2050 us).
//
// Fragment layout (16x16x128): lane l supplies row l % 16 and, with g = l / 16, the bytes
// [16 g, +16) and [64 + 16 g, +16) of the 128-wide K block. Accumulator register i of lane l
// is D[4 g + i][l % 16]: weight row 4 g + i of the fragment, token l % 16.
#include <type_traits>

#include "gemm_mid.h"
#include "mapping.h"
#include "moe_common.h"
#include "moe_internal.h"

namespace moe {

constexpr int kMidCols = 256;
constexpr int kMidThreads = 256;
constexpr int kMidMaxKB = 128;  // K <= 16384

struct MidLds {
  uint8_t* b;         // weight tile: 256 rows x 128 bytes
  uint8_t* a;         // token rows: two buffers of TR x 128 bytes (TR: 64 or 128 tile rows)
  uint8_t* sa;        // activation scales: two buffers of TR rows x 4 K blocks; at the end the
                      // last block scale per (half, row)
  float (*sw)[kMidMaxKB];
  int* tok;           // token (gate_up) or h row (down) of each tile row; -1: none
  float* r;           // scale ratios [step & 1][half][row]; at the end the waves' row maxima [4][row]
};

// LDS reads left in flight (lds_read16) until a wait names their registers.
template <int OFF>
__device__ __forceinline__ void mid_read4(uint32_t addr, float& v) {
  asm volatile("ds_read_b32 %0, %1 offset:%2" : "=&v"(v) : "v"(addr), "n"(OFF) : "memory");
}
// A token fragment (16 rows) and the lane's token's scale ratios (gate_up: gate and up half;
// down: the wave's half), or its scale in r0.
struct MidFragA {
  v4i lo, hi;
  float r0, r1;
};
template <bool RATIO, int N = 0>  // all but the newest N LDS reads
__device__ __forceinline__ void mid_wait(MidFragA& f) {
  if constexpr (RATIO)
    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(f.lo), "+v"(f.hi), "+v"(f.r0), "+v"(f.r1) : "n"(N) : "memory");
  else
    asm volatile("s_waitcnt lgkmcnt(%3)" : "+v"(f.lo), "+v"(f.hi), "+v"(f.r0) : "n"(N) : "memory");
}
template <int N>
__device__ __forceinline__ void mid_wait_b(v4i (&b)[8], float& s0, float& s1) {
  asm volatile("s_waitcnt lgkmcnt(%10)"
               : "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]), "+v"(b[4]), "+v"(b[5]), "+v"(b[6]),
                 "+v"(b[7]), "+v"(s0), "+v"(s1)
               : "n"(N)
               : "memory");
}
// Token fragment m from token buffer BUF: with ratios, those of the two halves (r_addr: the
// ratios); otherwise the tokens' scales of K block Q of the group (r_addr: the group's).
template <int KIND, int TR, int BUF, int Q, bool RATIO>
__device__ __forceinline__ void mid_read_a(uint32_t lo, uint32_t hi, uint32_t r_addr, int m, MidFragA& f) {
#define MID_A(M)                                                                \
  case M:                                                                       \
    lds_read16<128 * TR * BUF + 2048 * M>(lo, f.lo);                            \
    lds_read16<128 * TR * BUF + 2048 * M>(hi, f.hi);                            \
    if constexpr (RATIO) {                                                      \
      mid_read4<8 * TR * BUF + 64 * M>(r_addr, f.r0);                           \
      mid_read4<8 * TR * BUF + 64 * M + (KIND == 0 ? 4 * TR : 0)>(r_addr, f.r1); \
    } else {                                                                    \
      mid_read4<256 * M + 4 * Q>(r_addr, f.r0);                                 \
    }                                                                           \
    break;
  switch (m) { MID_A(0) MID_A(1) MID_A(2) MID_A(3) MID_A(4) MID_A(5) MID_A(6) MID_A(7) }
#undef MID_A
}

__device__ __forceinline__ v8i mid_cat(const v4i& lo, const v4i& hi) {
  return (v8i){lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
}
__device__ __forceinline__ v4f mid_mfma(const v8i& w, const v8i& t, const v4f& c) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, t, c, 0, 0, 0, 0, 0, 0);
}

// One work item: rows [slot0, slot0 + nrows) of expert e (hq / y rows from rbase), at most
// 16 MF of them, against column tile nt; alone: e has no
// other row tile.
template <int KIND, int TR, int MF, bool RATIO>
__device__ __forceinline__ void mid_item(const MidArgs& p, const MidLds& s, const int e, const long slot0,
                                         const long rbase, const int nrows, const int nt, const bool alone) {
  constexpr int NA = (MF + 1) / 2;       // token-row loads per wave and step
  // Token fragments in registers, read D - 1 ahead (from seven row groups on the accumulators
  // leave room for two).
  constexpr int D = TR > 64 && MF <= 6 ? 3 : 2;
  constexpr int kA = TR * 128, kS = TR * 16;  // bytes of a token and of a scale buffer
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r16 = lane & 15;
  const int Kdim = (KIND == 0) ? p.H : p.I;
  const int KB = Kdim / 128;  // a multiple of 4
  const int rows_w = (KIND == 0) ? 2 * p.I : p.H;
  const bool is_sh = e >= p.E;
  const int ej = is_sh ? e - p.E : e;
  const long arows = (KIND == 0) ? p.T : p.rows;
  const buf_rsrc_t rw = buf_rsrc((is_sh ? p.wsh : p.w) + (size_t)ej * rows_w * Kdim, (long)rows_w * Kdim);
  const buf_rsrc_t ra = buf_rsrc(p.a, arows * Kdim);
  const buf_rsrc_t rs = buf_rsrc(p.as, arows * KB * 4);
  const float* const wsb = (is_sh ? p.wssh : p.ws) + (size_t)ej * (rows_w / 128) * KB;

  // Tile row -> weight row. Wave w multiplies gate rows 32 w .. + 31 and the matching up
  // rows (tile rows 128 on), or 64 outputs. Row 16 n + 4 g + i of a wave's part holds output
  // column 8 g + 4 n + i (gate_up) or 16 g + 4 n + i (down).
  auto wrow_of = [&](int row) -> int {
    const int gi = row & 15;
    if (KIND == 0) {
      const int hc = nt * 128 + (row & 96) + 8 * (gi >> 2) + 4 * ((row >> 4) & 1) + (gi & 3);
      return row < 128 ? hc : p.I + hc;
    }
    return nt * kMidCols + (row & 192) + 16 * (gi >> 2) + 4 * ((row >> 4) & 3) + (gi & 3);
  };
  // Weight loads: wave w fills tile rows [64 w, +64), load i rows 64 w + 8 i + l / 8,
  // stored chunk l % 8 = logical chunk swz(row, l % 8).
  uint32_t boff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 64 * wave + 8 * i + (lane >> 3);
    boff[i] = (uint32_t)wrow_of(row) * (uint32_t)Kdim + (uint32_t)(swz(row, lane & 7) * 16);
  }
  // An expert of one tile reads its weights once: non-temporal, so the stream leaves the
  // token rows in L2; sibling tiles share them through L2.
  auto load_b = [&](int kb) {
    auto one = [&](int i, auto nt_c) {
      const int q = i >> 1, drow = KIND == 0 ? 4 * (q & 1) + 32 * (q >> 1) : 4 * q;  // rows past boff's
      buf_lds16<decltype(nt_c)::value>(rw, boff[i & 1], drow * Kdim + kb * 128, s.b + (8 * wave + i) * 1024);
    };
    if (alone) {
#pragma unroll
      for (int i = 0; i < 8; ++i) one(i, std::true_type{});
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) one(i, std::false_type{});
    }
  };
  // Token (gate_up) or h row (down) behind a tile row; rows with none read row 0 and are
  // not stored. Ids first: the token rows' addresses need them, and loads return in order.
  auto id_of = [&](int row) -> int {
    if (KIND == 1) return (int)rbase + row;
    if (is_sh) return (int)(slot0 - p.NB - (long)ej * p.T) + row;
    return p.tpid[slot0 + min(row, nrows - 1)];
  };
  auto src_of = [&](int row, int id) -> int {
    return (row < nrows && id >= 0 && (KIND == 1 || id < p.T)) ? id : -1;
  };
  int areg[NA], aid[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    areg[i] = min(wave + 4 * i, 2 * MF - 1);  // 8-row region; past the last, the last once more
    aid[i] = id_of(8 * areg[i] + (lane >> 3));
  }
  const int srow = TR > 64 ? 64 * (wave & 1) + lane : lane;  // waves below TR / 64 load the scales
  const int sid = id_of(srow);
  __builtin_amdgcn_sched_barrier(0);
  load_b(0);
  __builtin_amdgcn_sched_barrier(0);
  uint32_t aoff[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int row = 8 * areg[i] + (lane >> 3), src = src_of(row, aid[i]);
    aoff[i] = (uint32_t)(src < 0 ? 0 : src) * (uint32_t)Kdim + (uint32_t)(swz(row, lane & 7) * 16);
  }
  const int ssrc = src_of(srow, sid);
  const uint32_t soff = (uint32_t)(ssrc < 0 ? 0 : ssrc) * (uint32_t)(KB * 4);
  auto load_a = [&](int i, int kb, int buf) {
    buf_lds16(ra, aoff[i], kb * 128, s.a + buf * kA + areg[i] * 1024);
  };
  auto load_s = [&](int grp) { buf_lds16(rs, soff, grp * 16, s.sa + (grp & 1) * kS + wave * 1024); };
#pragma unroll
  for (int i = 0; i < NA; ++i) load_a(i, 0, 0);
  if (wave < TR / 64) {
    load_s(0);
    lds_st32(lds_addr(s.tok) + 4 * srow, ssrc);
  }
  // weight block scales of the tile's two 128-row halves (gate / up, or two output blocks)
  for (int i = tid; i < 2 * KB; i += kMidThreads) {
    const int h = i < KB ? 0 : 1, kb = i - h * KB;
    const int rb = (KIND == 0) ? (h == 0 ? nt : p.I / 128 + nt) : nt * 2 + h;
    lds_st32(lds_addr(&s.sw[h][kb]), __float_as_int(wsb[(size_t)rb * KB + kb]));
  }

  v4f acc[MF][4];
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int n = 0; n < 4; ++n) acc[m][n] = (v4f){0.f, 0.f, 0.f, 0.f};

  const uint32_t sw = (r16 >> 1) & 7;
  const uint32_t b_base = lds_addr(s.b) + ((KIND == 0 ? 32 : 64) * wave + r16) * 128;
  const uint32_t b_lo = b_base + ((g ^ sw) << 4), b_hi = b_base + (((4 + g) ^ sw) << 4);
  const uint32_t a_lo = lds_addr(s.a) + r16 * 128 + ((g ^ sw) << 4);
  const uint32_t a_hi = lds_addr(s.a) + r16 * 128 + (((4 + g) ^ sw) << 4);
  const uint32_t sa_base = lds_addr(s.sa) + r16 * 16;
  const uint32_t w0_base = lds_addr(&s.sw[KIND == 0 ? 0 : wave >> 1][0]);
  const uint32_t w1_base = lds_addr(&s.sw[KIND == 0 ? 1 : wave >> 1][0]);
  const uint32_t r_base = lds_addr(s.r) + 4 * r16 + (KIND == 1 ? 4 * TR * (wave >> 1) : 0);
  // Scale ratios (TR = 128): lane j of wave w owns row 64 (w % 2) + j of half w / 2 and writes
  // block k + 1's during step k. Rows without a source use scale 1; a zero scale (an all-zero weight block,
  // whose products are zero) repeats the previous one.
  const int orow = 64 * (wave & 1) + lane, ohalf = wave >> 1;
  const uint32_t osa = lds_addr(s.sa) + 16 * orow;
  const uint32_t osw = lds_addr(&s.sw[ohalf][0]);
  const uint32_t odst = lds_addr(s.r) + 4 * (TR * ohalf + orow);
  float s_prev = 0.f;
  bool ovalid = false;
  auto ratio = [&](float sa, float sw) {
    float sc = ovalid ? sa * sw : 1.f;
    if (sc == 0.f) sc = (s_prev != 0.f) ? s_prev : 1.f;
    const float r = s_prev / sc;
    s_prev = sc;
    return r;
  };

  // Step kb = 4 grp + Q. Everything of step kb + 1 is loaded meanwhile.
  auto step = [&](int grp, auto q_c, bool more) {
    constexpr int Q = decltype(q_c)::value, BUF = Q & 1;
    const int kb = 4 * grp + Q;
    wait_vm<0>();   // the step's tiles and scales have landed
    lds_barrier();  // ... for every wave, and its ratios are written
    v4i b[8];
    float nsa, nsw;
    MidFragA f[D];
    constexpr int r1 = 16, r2 = KIND == 0 ? 128 : 32, r3 = KIND == 0 ? 144 : 48;
    lds_read16<0>(b_lo, b[0]);
    lds_read16<0>(b_hi, b[1]);
    lds_read16<r1 * 128>(b_lo, b[2]);
    lds_read16<r1 * 128>(b_hi, b[3]);
    lds_read16<r2 * 128>(b_lo, b[4]);
    lds_read16<r2 * 128>(b_hi, b[5]);
    lds_read16<r3 * 128>(b_lo, b[6]);
    lds_read16<r3 * 128>(b_hi, b[7]);
    // ratios: the next block's scales (past the last block: not used); otherwise this block's
    // weight scales of the wave's gate and up (or output) half
    if constexpr (RATIO) {
      mid_read4<4 * ((Q + 1) & 3)>(osa + ((grp + (Q == 3)) & 1) * kS, nsa);
      mid_read4<4 * (Q + 1)>(osw + 16 * grp, nsw);
    } else {
      mid_read4<4 * Q>(w0_base + 16 * grp, nsa);
      mid_read4<4 * Q>(w1_base + 16 * grp, nsw);
    }
    const uint32_t ra0 = RATIO ? r_base : sa_base + (grp & 1) * kS;
    mid_read_a<KIND, TR, BUF, Q, RATIO>(a_lo, a_hi, ra0, 0, f[0]);
    mid_wait_b<RATIO ? 4 : 3>(b, nsa, nsw);
    lds_barrier();  // every wave holds its weight fragments
    if (more) {
#pragma unroll
      for (int i = 0; i < NA; ++i) load_a(i, kb + 1, BUF ^ 1);
      load_b(kb + 1);
      if (Q == 0 && wave < TR / 64) load_s(grp + 1);  // past the last group: not used
      if constexpr (RATIO) lds_st32(odst + 8 * TR * (BUF ^ 1), __float_as_int(ratio(nsa, nsw)));
    }
    if (D > 2 && MF > 1) mid_read_a<KIND, TR, BUF, Q, RATIO>(a_lo, a_hi, ra0, 1, f[1]);
    mid_wait<RATIO, (D > 2 && MF > 1) ? 4 : 0>(f[0]);
    if constexpr (!RATIO) {
      // fragment m's four products, scaled and added (the other workgroups' waves fill the wait)
#pragma unroll
      for (int m = 0; m < MF; ++m) {
        if (m + 1 < MF) mid_read_a<KIND, TR, BUF, Q, RATIO>(a_lo, a_hi, ra0, m + 1, f[(m + 1) & 1]);
        const v8i t = mid_cat(f[m & 1].lo, f[m & 1].hi);
        const float c0 = f[m & 1].r0 * nsa, c1 = f[m & 1].r0 * nsw;
        v4f part[4];
#pragma unroll
        for (int n = 0; n < 4; ++n)
          part[n] = mid_mfma(mid_cat(b[2 * n], b[2 * n + 1]), t, (v4f){0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[m][n] += part[n] * ((KIND == 0 && n >= 2) ? c1 : c0);
        acc_pin(acc[m]);
        if (m + 1 < MF) mid_wait<RATIO>(f[(m + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
      return;
    }
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      if (m + D - 1 < MF) mid_read_a<KIND, TR, BUF, Q, RATIO>(a_lo, a_hi, ra0, m + D - 1, f[(m + D - 1) % D]);
      const MidFragA& x = f[m % D];
      const v8i t = mid_cat(x.lo, x.hi);
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        __builtin_amdgcn_sched_barrier(0);
        acc[m][n] = mid_mfma(mid_cat(b[2 * n], b[2 * n + 1]), t, acc[m][n] * ((KIND == 0 && n >= 2) ? x.r1 : x.r0));
        __builtin_amdgcn_sched_barrier(0);
      }
      acc_pin(acc[m > 0 ? m - 1 : MF - 1]);
      if (m + 1 < MF) {
        if (D > 2 && m + 2 < MF)
          mid_wait<RATIO, 4>(f[(m + 1) % D]);
        else
          mid_wait<RATIO>(f[(m + 1) % D]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // the first block's ratios (s_prev = 0: the accumulators start at 0)
  if constexpr (RATIO) {
    wait_vm<0>();
    lds_barrier();
    float fsa, fsw;
    int valid;
    asm volatile("ds_read_b32 %0, %3\n\tds_read_b32 %1, %4\n\tds_read_b32 %2, %5\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(fsa), "=&v"(fsw), "=&v"(valid)
                 : "v"(osa), "v"(osw), "v"(lds_addr(s.tok) + 4 * orow)
                 : "memory");
    ovalid = valid >= 0;
    lds_st32(odst, __float_as_int(ratio(fsa, fsw)));
  }
  for (int grp = 0; grp < KB / 4; ++grp) {
    step(grp, std::integral_constant<int, 0>{}, true);
    step(grp, std::integral_constant<int, 1>{}, true);
    step(grp, std::integral_constant<int, 2>{}, true);
    step(grp, std::integral_constant<int, 3>{}, grp + 1 < KB / 4);
  }

  // Epilogue: lane l holds token row 16 m + l % 16.
  __syncthreads();  // the last step's reads are done: its scale and ratio buffers are reused
  float* const last = (float*)s.sa;
  if constexpr (RATIO) {
    last[TR * ohalf + orow] = s_prev;
    __syncthreads();
  }
  // per-output-channel weight scales, 1 when absent (a multiply by 1 is exact)
  const float* const csb = RATIO ? nullptr : is_sh ? p.cssh : p.cs;
  auto chan = [&](int row) { return csb == nullptr ? 1.f : csb[(size_t)ej * rows_w + row]; };
  if (KIND == 0) {
    // h = SiLU(gate) * up for 8 consecutive h columns; the row maximum of the 1x128 group is
    // combined over the four lanes of the token and the four waves
    const int hc = nt * 128 + 32 * wave + 8 * g;
    float cg[8], cu[8];
    if constexpr (!RATIO) {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        cg[c] = chan(hc + c);
        cu[c] = chan(p.I + hc + c);
      }
    }
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      const float sg_ = RATIO ? last[16 * m + r16] : 1.f, su = RATIO ? last[TR + 16 * m + r16] : 1.f;
      float mx = 0.f;
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float gt = acc[m][n][i] * (RATIO ? sg_ : cg[4 * n + i]);
          const float up = acc[m][n + 2][i] * (RATIO ? su : cu[4 * n + i]);
          // hardware reciprocal (about 1 ulp): h only feeds the 1x128 fp8 quantization
          const float h = gt * __builtin_amdgcn_rcpf(1.0f + __expf(-gt)) * up;
          acc[m][n][i] = h;
          mx = fmaxf(mx, fabsf(h));
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      if (g == 0) s.r[TR * wave + 16 * m + r16] = mx;
    }
    __syncthreads();
    const int GI = p.I / 128;
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      const int row = 16 * m + r16;
      const float amax = fmaxf(fmaxf(s.r[row], s.r[TR + row]),
                               fmaxf(s.r[2 * TR + row], s.r[3 * TR + row]));
      const float sc = fmaxf(amax, 0x1.b7cdfep-34f) / 448.0f;
      const float rsc = 1.0f / sc;
      uint32_t c[2];
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = fminf(fmaxf(div_by(acc[m][n][i], sc, rsc), -448.0f), 448.0f);
        c[n] = e4m3x2(v[0], v[1]) | (e4m3x2(v[2], v[3]) << 16);
      }
      if (row < nrows && s.tok[row] >= 0) {
        *(uint2*)(p.hq + (size_t)(rbase + row) * p.I + hc) = make_uint2(c[0], c[1]);
        if (wave == 0 && g == 0) p.hs[(size_t)(rbase + row) * GI + nt] = sc;
      }
    }
  } else {
    const int oc = nt * kMidCols + 64 * wave + 16 * g;
    float co[16];
    if constexpr (!RATIO) {
#pragma unroll
      for (int c = 0; c < 16; ++c) co[c] = chan(oc + c);
    }
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      const int row = 16 * m + r16;
      const float sl = RATIO ? last[TR * (wave >> 1) + row] : 1.f;
      int o[8];
#pragma unroll
      for (int n = 0; n < 4; ++n)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          o[2 * n + i] = (int)bf16x2(acc[m][n][2 * i] * (RATIO ? sl : co[4 * n + 2 * i]),
                                     acc[m][n][2 * i + 1] * (RATIO ? sl : co[4 * n + 2 * i + 1]));
      if (row < nrows) {
        int4* const y = (int4*)(p.y + (size_t)(rbase + row) * p.H + oc);
        y[0] = make_int4(o[0], o[1], o[2], o[3]);
        y[1] = make_int4(o[4], o[5], o[6], o[7]);
      }
    }
  }
}

// TR = 128: the block kernels' arithmetic on block tiles; 64: the row-tile kernels' on row tiles.
template <int KIND, int TR>
__global__ __launch_bounds__(kMidThreads, TR > 64 ? 2 : 3) void expert_gemm_mid_kernel(MidArgs p) {
  constexpr bool RATIO = TR > 64;
  __shared__ __attribute__((aligned(1024))) uint8_t sB[kMidCols * 128];
  __shared__ __attribute__((aligned(1024))) uint8_t sA[2 * TR * 128];
  __shared__ __attribute__((aligned(1024))) uint8_t sSA[2 * TR * 16];
  __shared__ float sW[2][kMidMaxKB];
  __shared__ int sTok[TR];
  __shared__ float sR[4 * TR];
  const MidLds s{sB, sA, sSA, sW, sTok, sR};
  const int NT = (KIND == 0) ? p.I / 128 : p.H / kMidCols;
  int tile, nt;
  bool alone;
  if constexpr (RATIO) {
    // XCD-aware item index, as in the block kernels
    const int x = blockIdx.x & 7;
    const int L = p.num_tiles[1 + x] * NT + (int)(blockIdx.x >> 3);
    if (L >= p.num_tiles[2 + x] * NT) return;
    const int2 sg = p.seg[L / NT];
    const int r0 = L - NT * sg.x;
    nt = r0 / sg.y;
    tile = sg.x + (r0 - nt * sg.y);
    alone = sg.y == 1;
    if (tile >= p.num_tiles[0]) return;  // truncated tile list
  } else {
    tile = blockIdx.x / NT;
    nt = blockIdx.x - tile * NT;
    const int n = p.num_tiles[0];
    if (tile >= n) return;
    const int e = p.tiles[tile].x;
    alone = (tile == 0 || p.tiles[tile - 1].x != e) && (tile + 1 >= n || p.tiles[tile + 1].x != e);
  }
  // (wave-uniform, so the operand bases stay in scalar registers)
  const int4 tv = p.tiles[tile];
  const int4 td = make_int4(__builtin_amdgcn_readfirstlane(tv.x), __builtin_amdgcn_readfirstlane(tv.y),
                            __builtin_amdgcn_readfirstlane(tv.z), __builtin_amdgcn_readfirstlane(tv.w));
  const int e = td.x, nrows = td.z;
  if (e < 0 || e >= p.E + p.nsh || nrows <= 0 || nrows > TR) return;
#define MID_ITEM(MF) return mid_item<KIND, TR, MF, RATIO>(p, s, e, td.y, td.w, nrows, nt, alone)
  if constexpr (TR > 64) {
    switch ((nrows + 15) / 16) {
      case 5: MID_ITEM(5);
      case 6: MID_ITEM(6);
      case 7: MID_ITEM(7);
      case 8: MID_ITEM(8);
    }
  }
  switch ((nrows + 15) / 16) {
    case 1: MID_ITEM(1);
    case 2: MID_ITEM(2);
    case 3: MID_ITEM(3);
    default: MID_ITEM(4);
  }
#undef MID_ITEM
}

bool mid_fits(int kind, const MidArgs& a) {
  auto al = [](const void* q, uintptr_t n) { return ((uintptr_t)q & (n - 1)) == 0; };
  const unsigned long lim = 1UL << 32;
  return a.H % 512 == 0 && a.I % 512 == 0 && a.H <= 128 * kMidMaxKB && a.I <= 128 * kMidMaxKB &&
         al(a.a, 16) && al(a.as, 16) && al(a.w, 16) && al(a.wsh, 16) && al(a.hq, 8) && al(a.y, 16) &&
         (unsigned long)(kind == 0 ? a.T : a.rows) * (unsigned long)(kind == 0 ? a.H : a.I) < lim &&
         2UL * a.I * a.H < lim && a.rows < (1L << 31);
}

template <int TR>
static void launch_mid_tiles(int kind, const MidArgs& a, long items, hipStream_t st) {
  const dim3 grid((unsigned)items), block(kMidThreads);
  if (kind == 0)
    hipLaunchKernelGGL((expert_gemm_mid_kernel<0, TR>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((expert_gemm_mid_kernel<1, TR>), grid, block, 0, st, a);
}

void launch_mid(int kind, const MidArgs& a, int max_tiles, hipStream_t st) {
  const long NT = (kind == 0) ? a.I / 128 : a.H / kMidCols;
  if (a.seg == nullptr)
    launch_mid_tiles<kMidTileRows>(kind, a, (long)max_tiles * NT, st);
  else  // each XCD's share of the block tiles
    launch_mid_tiles<kMidTallRows>(kind, a, 8L * block_tiles_cap(max_tiles) * NT, st);
}

}  // namespace moe

using namespace moe;

int moe::mid_max_tiles(int T, int K, int E, int n_shared) {
  const long rows = (long)T * std::min(K, E);
  return (int)(rows / kMidTallRows + std::min<long>(E, rows) +
               (long)n_shared * ((T + kMidTallRows - 1) / kMidTallRows));
}
