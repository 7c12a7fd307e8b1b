// 2 .. 16 rows through a matrix of 4-bit codes that lie along K (q4f16_1, AutoGPTQ), activations in registers.
//
// The ring kernel (skinny_gemm.h) takes the activations through LDS once per 16 .. 128 columns and makes every weight in packed
// fp16.  Here a workgroup per CU walks over tiles of 16 columns, its 8 wavefronts split K into contiguous runs of PW
// pieces (256 k, 128 bytes of a column), and a wavefront keeps the activations of its run as MFMA operands for the whole kernel.
// In the walk there are only the codes, which go from memory to the registers that feed the products (whole lines, 8
// columns x 128 bytes a load, the next tile's requested as soon as a register has been read), and a tile's scales, fetched
// by all wavefronts for one another a tile ahead and kept in LDS.  Per tile the 8 partial sums meet in LDS; wavefronts take turns
// at adding them up.
//
// What bounds it: with many tiles the weight stream (N = 28672, K = 8192, M = 3 / 8 4.9 / 4.6 TB/s) and, from 9 rows on, the vector
// unit (M = 16 3.6 TB/s: exchange of halves, lane swaps and 4 fmas a product); with few the prologue, in which all activations
// come from L2 (3 us at M = 8, K = 4096), and about 0.5 us a tile of meeting and adding.
//
// Products.  A weight is not made: codes become fp16 numbers by masks alone (the code in bits 0 .. 3 of a half is the number
// 2^-24 q, in bits 4 .. 7 2^-20 q; the activations of the former are taken 16 times), a product holds codes of one scale
// group, and zero point and scale are applied to its result in fp32:
//   q4f16_1   one v_mfma_f32_16x16x32_f16 per group, which begins at -7 times the sum of the group's activations; the words of
//             a group are spread over the four lane quarters by two lane swaps for two words;
//   AutoGPTQ  (group size a multiple of 128) the four products of 128 k as the words come, then minus the zero point times the
//             sum of the activations.
// Up to 8 rows (HALF) the 16 rows of the operand hold each of them twice, at the k of the two halves of a piece, so that what
// a load brings (8 columns, two halves) are the columns of one product as they come; results of a row half against the
// other column half are sums of nothing and dropped.  With more rows two loads exchange halves first.
// Activations of 4094 and more, infinite ones and NaN (16 times them is no number, or the sum that is taken off is not what
// the products hold) take weights as the formats define them, rounded to fp16: in every row, in the wavefronts whose run holds
// one.  The codes come as ever, but the vector unit makes the weights: with such an activation in every run N = 22016, K = 4096 takes
// 19.1 / 20.7 / 23.9 us at M = 3 / 8 / 16 in place of 13.8 / 14.6 / 17.1, N = 28672, K = 8192 37.1 / 40.2 / 46.5 in place of
// 27.9 / 29.9 / 36.3 (25.2 / 26.9 / 30.8 and 57.5 / 60.9 / 67.3 where those wavefronts fetched a tile's codes once more and
// waited for them).  Rounded weights of a row's own would need two sets of operands, which the registers do not hold; with
// rows at 1/16 of their factor a weight of exactly 0 leaves 2^-17 of its two products.
#ifndef RELAX_AMD_CSRC_HELD_GEMM_H_
#define RELAX_AMD_CSRC_HELD_GEMM_H_

#include <type_traits>

#include "code_products.h"
#include "tuning.h"
#include "wq_device.h"
#include "wq_host.h"

namespace wq {

struct HeldArgs {
  const char* W;       // [N, K/2] bytes
  const char* S;       // q4f16_1: fp16 [N, K/32]; AutoGPTQ: (scale, zero point + 1) [N, groups]
  int groups;          // AutoGPTQ: groups per column
  int group128;        // ... and 128-k chunks per group
};

enum HeldFormat { kHeldQ4, kHeldGptq };

template <HeldFormat FMT, int MODE, int PW>
struct HeldCfg {
  static constexpr bool kHalf = MODE == 0;             // up to 8 rows
  static constexpr int kOps = kHalf ? 4 : 8;           // operands per piece
  static constexpr int kDepth = PW <= 2 ? 2 : 1;       // tiles whose codes are on their way
  static constexpr int kWords = FMT == kHeldQ4 ? 32 * PW : 16 * PW;  // 4-byte words of scales per column in LDS
  static constexpr int kLoads = FMT == kHeldQ4 ? PW : (PW + 1) / 2;  // loads of them per wavefront and tile (two columns)
  static constexpr int kColBytes = FMT == kHeldQ4 ? kWords * 4 + 16 : (kWords | 1) * 4;  // (columns on different banks)
  static constexpr int kScaleBytes = 16 * kColBytes;
  static constexpr int kPartBytes = kHalf ? 512 : 1024;
  static constexpr int kLdsBytes = 2 * kScaleBytes + 16 * kPartBytes;
  // start values of the products in registers, where there is room
  static constexpr bool kKeep = FMT == kHeldQ4 && (kHalf ? PW <= 4 : PW <= 2);
  // AutoGPTQ: the sums of activations, the same for all 16 columns, one per lane of 16 instead of all in every lane
  static constexpr bool kPackSums = FMT == kHeldGptq && !kHalf && PW == 4;
};

// v of lane n of every 16
__device__ __forceinline__ float row_broadcast(float v, int n) {
#define WQ_ROW_BROADCAST(N) \
  case N: return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150 + N /* row_newbcast */, 0xf, 0xf, false))
  switch (n) {
    WQ_ROW_BROADCAST(0);
    WQ_ROW_BROADCAST(1);
    WQ_ROW_BROADCAST(2);
    WQ_ROW_BROADCAST(3);
    WQ_ROW_BROADCAST(4);
    WQ_ROW_BROADCAST(5);
    WQ_ROW_BROADCAST(6);
    default:
    WQ_ROW_BROADCAST(7);
  }
#undef WQ_ROW_BROADCAST
}

template <HeldFormat FMT, int MODE, int PW, class Epilogue>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void held_gemm_kernel(HeldArgs args, const half_t* __restrict__ X, half_t* __restrict__ Y, Epilogue epi, int M, int N, int K) {
  using Cfg = HeldCfg<FMT, MODE, PW>;
  constexpr bool HALF = Cfg::kHalf;
  constexpr int D = Cfg::kDepth, NO = Cfg::kOps, NL = Cfg::kLoads, COL = Cfg::kColBytes, PART = Cfg::kPartBytes;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int ks = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, kq = lane >> 4;
  const int tiles = (N + 15) >> 4, grid = gridDim.x;
  const int col_bytes = K >> 1, groups32 = K >> 5;
  unsigned char* const parts = lds + 2 * Cfg::kScaleBytes;
  constexpr uint32_t kOut = 0x80000000u;  // beyond every descriptor: brings zeros

  // ---- where a lane's codes and scales lie from a tile's first column on ----
  uint32_t w_off[PW];
#pragma unroll
  for (int p = 0; p < PW; ++p) {
    const int g = 8 * (ks * PW + p) + 4 * (i >> 3) + kq;
    w_off[p] = g < groups32 ? (uint32_t)((i & 7) * col_bytes + g * 16) : kOut;
  }
  const int s_col = FMT == kHeldQ4 ? groups32 * 2 : args.groups * 4;  // bytes of a column
  // (whole wavefronts per column: the second column's lie a column further)
  constexpr int NS = Cfg::kWords % 64 == 0 ? NL / 2 : NL;
  uint32_t s_off[NS], s_to[NS];
  auto scale_from = [&](int t) { return s_off[t % NS] + (uint32_t)(t / NS * s_col); };  // (beyond every descriptor stays there)
  auto scale_to = [&](int t) { return s_to[t % NS] + (uint32_t)(t / NS * COL); };
#pragma unroll
  for (int t = 0; t < NS; ++t) {
    const int idx = t * 64 + lane, c = idx / Cfg::kWords, d = idx % Cfg::kWords;  // column of the wavefront's two, word
    const bool held = c < 2 && (FMT == kHeldQ4 ? 2 * d < groups32 : 128 * d < K);
    const int at = FMT == kHeldQ4 ? 4 * d : 4 * (d / args.group128);
    s_off[t] = held ? (uint32_t)((2 * ks + c) * s_col + at) : kOut;
    s_to[t] = (uint32_t)(min(2 * ks + c, 15) * COL + d * 4);
  }
  auto tile_rows = [&](int tile) { return max(min(16, N - tile * 16), 0); };  // 0 past the last tile: empty descriptors
  struct Codes {
    wq_rsrc_t half[2];  // columns 0 .. 7 and 8 .. 15 (those that are not there bring zeros)
  };
  auto codes_at = [&](int tile) {
    const int rows = tile_rows(tile), first = __builtin_amdgcn_readfirstlane(min(rows, 8)), second = __builtin_amdgcn_readfirstlane(rows) - first;
    const char* const from = args.W + (int64_t)min(tile, tiles - 1) * 16 * col_bytes;
    return Codes{{wq_rsrc(from, first * col_bytes), wq_rsrc(from + first * col_bytes, second * col_bytes)}};
  };
  auto scales_at = [&](int tile) {
    return wq_rsrc(args.S + (int64_t)min(tile, tiles - 1) * 16 * s_col, __builtin_amdgcn_readfirstlane(tile_rows(tile) * s_col));
  };
  auto request = [&](const Codes& from, int p, int h) {
    return __builtin_amdgcn_raw_buffer_load_b128(from.half[h], w_off[p], 0, 2 /* nt */);
  };

  // ---- everything that the first tile needs is requested at once: activations, scales of two tiles, codes ----
  half8_t xb[PW][NO];  // operand o of piece p
  uint4_t raw[PW][NO];
  auto fetch_x = [&]() {
    const wq_rsrc_t xr = wq_rsrc(reinterpret_cast<const char*>(X), 2 * M * K);
#pragma unroll
    for (int p = 0; p < PW; ++p)
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        // Whole lines, 8 rows x 128 bytes a load, for two operands o, o + 1: q4f16_1 takes dword kq of groups e, e + 1
        // from 64 bytes each, AutoGPTQ dwords e, e + 1 of the 32 codes of quarter kq.  Up to 8 rows the two loads are the two
        // halves of the piece, with more they are rows 0 .. 7 and 8 .. 15.
        const int second = o & 1, e = (o & 3) - second, row = min((i & 7) + (HALF ? 0 : 8 * second), M - 1);
        const int k = 256 * (ks * PW + p) + 128 * (HALF ? second : o >> 2) +
                      (FMT == kHeldQ4 ? 32 * (e + (i >> 3)) + 8 * kq : 32 * kq + 8 * (e + (i >> 3)));
        raw[p][o] = __builtin_amdgcn_raw_buffer_load_b128(xr, k < K ? (uint32_t)(row * K + k) * 2u : kOut, 0, 0);
      }
    __builtin_amdgcn_sched_barrier(0);
  };
  fetch_x();
  uint4_t word[D][2 * PW];
  uint32_t sw[NL], sw0[NL];
  auto fetch_scales = [&](int tile, uint32_t (&to)[NL]) {
    const wq_rsrc_t from = scales_at(tile);
#pragma unroll
    for (int t = 0; t < NL; ++t) to[t] = __builtin_amdgcn_raw_buffer_load_b32(from, scale_from(t), 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto put_scales = [&](int buf, const uint32_t (&from)[NL]) {
#pragma unroll
    for (int t = 0; t < NL; ++t)
      if ((t + 1) * 64 <= 2 * Cfg::kWords || t * 64 + lane < 2 * Cfg::kWords) *reinterpret_cast<uint32_t*>(lds + buf * Cfg::kScaleBytes + scale_to(t)) = from[t];
  };
  int tile = blockIdx.x;
  fetch_scales(tile, sw0);
  fetch_scales(tile + grid, sw);
#pragma unroll
  for (int a = 0; a < D; ++a) {
    const Codes from = codes_at(tile + a * grid);
#pragma unroll
    for (int l = 0; l < 2 * PW; ++l) {
      word[a][l] = request(from, l >> 1, l & 1);
      __builtin_amdgcn_sched_barrier(0);  // in this order everywhere: the waits count on it
    }
  }

  // ---- activations as operands ----
  float4_t start[Cfg::kKeep ? PW : 1][NO];      // q4f16_1: what the products begin at
  float4_t xsum[Cfg::kPackSums ? 1 : PW][HALF || Cfg::kPackSums ? 1 : 2];  // AutoGPTQ: sums over 128 k
  if constexpr (Cfg::kPackSums) xsum[0][0] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
  const uint4_t kSeven = {0x80078007u, 0x80708070u, 0x80078007u, 0x80708070u};
  const uint4_t kOne = {0x00010001u, 0x00100010u, 0x00010001u, 0x00100010u};
  const half8_t weigh = __builtin_bit_cast(half8_t, FMT == kHeldQ4 ? kSeven : kOne);
  auto sum_of = [&](const half8_t& a, const float4_t& c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, weigh, c, 0, 0, 0); };
  const float4_t kNull = {0.0f, 0.0f, 0.0f, 0.0f};
  // activations as operands; those of codes in bits 0 .. 3 times `low`
  auto build = [&](half_t low) {
    const half2_t l2 = {low, low};
#pragma unroll
    for (int p = 0; p < PW; ++p)
#pragma unroll
      for (int o = 0; o < NO; o += 2) {
        uint32_t in[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h) in[h][0] = raw[p][o + h].x, in[h][1] = raw[p][o + h].y, in[h][2] = raw[p][o + h].z, in[h][3] = raw[p][o + h].w;
        exchange_halves(in[0], in[1]);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          uint32_t q[4];
          pair_i_i4(in[h], q);
          xb[p][o + h] = __builtin_bit_cast(half8_t, uint4_t{as_u32(as_half2(q[0]) * l2), q[1], as_u32(as_half2(q[2]) * l2), q[3]});
        }
      }
  };
  build((half_t)16.0f);
  float zero = 0.0f;  // NaN where 16 times an activation is infinite or not a number
#pragma unroll
  for (int p = 0; p < PW; ++p) {
    float4_t c;
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      if constexpr (FMT == kHeldQ4) {
        c = sum_of(xb[p][o], kNull);
        if constexpr (Cfg::kKeep) start[p][o] = c;
      } else if constexpr (Cfg::kPackSums) {
        c = sum_of(xb[p][o], (o & 3) == 0 ? kNull : c);
        if ((o & 3) == 3) {
#pragma unroll
          for (int e = 0; e < 4; ++e) xsum[0][0][e] = i == 2 * p + (o >> 2) ? c[e] : xsum[0][0][e];
        }
      } else {
        c = sum_of(xb[p][o], (o & 3) == 0 ? kNull : xsum[p][o >> 2]);
        xsum[p][o >> 2] = c;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) zero = fmaf(c[e], 0.0f, zero);
    }
  }
  // (a number in a scalar register: as a lane mask it makes ways through the loop on which no loads are issued, and the compiler
  // waits for all that are on their way)
  const int special = __builtin_amdgcn_readfirstlane(__builtin_amdgcn_ballot_w64(zero != 0.0f) != 0 ? 1 : 0);
  if (special) {
    fetch_x();
    build((half_t)1.0f);
  }

  // a word of codes as weights rounded to fp16: (code - off) * s
  auto weights = [&](uint32_t w, half_t off, half_t s) {
    const half_t o = off + (half_t)1024.0f;
    const half2_t o2 = {o, o}, s2 = {s, s};
    uint32_t r[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) r[d] = as_u32((as_half2(((w >> (4 * d)) & 0x000F000Fu) | 0x64006400u) - o2) * s2);
    return __builtin_bit_cast(half8_t, uint4_t{r[0], r[1], r[2], r[3]});
  };
  auto arrange = [&](uint32_t (&w)[2][4]) {
    if constexpr (!HALF) exchange_halves(w[0], w[1]);
    if constexpr (FMT == kHeldQ4) {
      spread_words(w[0]);
      spread_words(w[1]);
    }
  };
  // scales of what w[h] holds after that: columns 0 .. 7, 8 .. 15 at the lane's half (HALF), or column i at half h
  auto scale_row = [&](int buf, int h) { return lds + buf * Cfg::kScaleBytes + (HALF ? 8 * h + (i & 7) : i) * COL; };

  constexpr int NA = HALF ? 2 : 1;
  auto multiply = [&](const Codes& next, uint4_t (&word)[2 * PW], int buf, float4_t (&acc)[NA]) {
#pragma unroll
    for (int p = 0; p < PW; ++p) {
      uint32_t w[2][4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        take_words(word[2 * p + h], w[h]);
        word[2 * p + h] = request(next, p, h);
      }
      arrange(w);
      float4_t t[2][2];
      if constexpr (FMT == kHeldQ4) {
        half4_t s4[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
          s4[h] = *reinterpret_cast<const half4_t*>(scale_row(buf, h) + (8 * (ks * PW + p) + 4 * (HALF ? i >> 3 : h)) * 2);
        // group by group, and behind the products the scaling of those of the group before
        auto scale = [&](int g) {
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[HALF ? h : 0][e] = fmaf(t[g & 1][h][e], (float)s4[h][g], acc[HALF ? h : 0][e]);
        };
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float4_t c[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int o = HALF ? g : 4 * h + g;
            if constexpr (Cfg::kKeep) c[h] = start[p][o];
            else if (HALF && h == 1) c[h] = c[0];
            else c[h] = sum_of(xb[p][o], kNull);
          }
#pragma unroll
          for (int h = 0; h < 2; ++h) t[g & 1][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xb[p][HALF ? g : 4 * h + g], code_operand(w[h][g]), c[h], 0, 0, 0);
          if (g > 0) scale(g - 1);
          __builtin_amdgcn_sched_barrier(0);
        }
        scale(3);
      } else {
        half2_t sz[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
          sz[h] = *reinterpret_cast<const half2_t*>(scale_row(buf, h) + (2 * (ks * PW + p) + (HALF ? i >> 3 : h)) * 4);
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            t[0][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xb[p][HALF ? d : 4 * h + d], code_operand(w[h][d]), d == 0 ? kNull : t[0][h], 0, 0, 0);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float x = Cfg::kPackSums ? row_broadcast(xsum[0][0][e], 2 * p + h) : xsum[Cfg::kPackSums ? 0 : p][HALF || Cfg::kPackSums ? 0 : h][e];
            const float v = fmaf(x, -(float)sz[h].y, t[0][h][e]);
            acc[HALF ? h : 0][e] = fmaf(v, (float)sz[h].x, acc[HALF ? h : 0][e]);
          }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // the same with rounded weights
  auto multiply_rounded = [&](const Codes& next, uint4_t (&word)[2 * PW], int buf, float4_t (&acc)[NA]) {
#pragma unroll
    for (int p = 0; p < PW; ++p) {
      uint32_t w[2][4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        take_words(word[2 * p + h], w[h]);
        word[2 * p + h] = request(next, p, h);
      }
      arrange(w);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          half_t off = (half_t)7.0f, s;
          if constexpr (FMT == kHeldQ4) {
            s = *reinterpret_cast<const half_t*>(scale_row(buf, h) + (8 * (ks * PW + p) + 4 * (HALF ? i >> 3 : h) + g) * 2);
          } else {
            const half2_t sz = *reinterpret_cast<const half2_t*>(scale_row(buf, h) + (2 * (ks * PW + p) + (HALF ? i >> 3 : h)) * 4);
            s = sz.x, off = sz.y;
          }
          const half8_t b = weights(w[h][g], off, s);
          acc[HALF ? h : 0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xb[p][HALF ? g : 4 * h + g], b, acc[HALF ? h : 0], 0, 0, 0);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[a] *= 1.0f / 1048576.0f;
  };

  // ---- the walk ----
  auto meet = [&]() {  // what this wavefront has written to LDS is visible to all, and they have read what they had to
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  put_scales(0, sw0);
  meet();
  auto step = [&](int j, uint4_t (&word)[2 * PW]) {
    const int buf = j & 1;
    const Codes next = codes_at(tile + D * grid);
    put_scales(buf ^ 1, sw);
    fetch_scales(tile + 2 * grid, sw);
    float4_t acc[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[a] = kNull;
    if (special) multiply_rounded(next, word, buf, acc);
    else multiply(next, word, buf, acc);
    // sums as [row][column] of the tile
    unsigned char* const set = parts + buf * 8 * PART;
    float* const part = reinterpret_cast<float*>(set + ks * PART);
    if constexpr (HALF) {
      float sum[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[e] = join_halves(acc[0][e], acc[NA - 1][e]);
      if (i < 8) {
#pragma unroll
        for (int e = 0; e < 4; ++e) part[(4 * (kq & 1) + e) * 16 + 8 * (kq >> 1) + i] = sum[e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) part[(4 * kq + e) * 16 + i] = acc[0][e];
    }
    meet();
    if (ks == (j & 7)) {
      constexpr int C = HALF ? 2 : 4;  // columns per lane
      const int m = HALF ? lane >> 3 : lane >> 2, c = (HALF ? lane & 7 : lane & 3) * C;
      float v[C];
#pragma unroll
      for (int e = 0; e < C; ++e) v[e] = 0.0f;
#pragma unroll
      for (int w = 0; w < 8; ++w)
#pragma unroll
        for (int e = 0; e < C; ++e) v[e] += reinterpret_cast<const float*>(set + w * PART)[m * 16 + c + e];
      if (m < M) {
#pragma unroll
        for (int e = 0; e < C; ++e) {
          const int n = tile * 16 + c + e;
          if (n < N) Y[(int64_t)m * N + n] = epi(v[e] * 1048576.0f, m, n);  // (the products were 2^-20 of themselves)
        }
      }
    }
    tile += grid;
  };
  int j = 0;
  for (; tile + (D - 1) * grid < tiles; j += D) {
#pragma unroll
    for (int a = 0; a < D; ++a) step(j + a, word[a]);
  }
  if constexpr (D == 2) {
    if (tile < tiles) step(j, word[0]);
  }
}

// pieces of 256 k that a wavefront's run has
inline int held_pieces(int64_t K) { return (int)(((K + 255) / 256 + 7) / 8); }
// the longest run whose activations fit the registers
inline int held_max_pieces(int64_t M) { return M <= 8 ? 5 : 4; }
inline bool held_fits(int64_t M, int64_t N, int64_t K) {
  return M >= 1 && M <= 16 && K % 64 == 0 && held_pieces(K) <= held_max_pieces(M) && 16 * K < (1ll << 30) && N < (1ll << 30);
}

// Where it is the faster one.  What it costs is that every workgroup loads all activations before its first tile and that its
// tiles go in whole rounds over the CUs; it pays from a few tiles per CU on, and with K long enough.
//   K > 4096, four tiles per CU or more: M = 3 / 8 / 16, N = 16384, K = 5120, q4f16_1 25.2 / 26.1 / 28.2 -> 13.9 / 14.8 / 18.7 us,
//     AutoGPTQ 24.7 / 25.6 / 27.8 -> 13.8 / 14.8 / 17.8; N = 28672, K = 8192 39.9 / 42.5 / 45.9 -> 27.0 / 29.0 / 36.2 and
//     38.2 / 40.2 / 43.5 -> 27.3 / 28.7 / 34.6.
//   Up to 8 rows, more than two: q4f16_1 from K = 4352 on (M = 8, N = 11008, K = 4608 12.8 -> 11.6, 8192 19.7 -> 15.9, 9728
//     23.6 -> 18.5; N = 8208, K = 4160 10.2 -> 10.6, N = 8192, K = 8192 12.2 -> 13.5), AutoGPTQ, whose ring kernel has more to
//     do per weight, from 3072 on (M = 8, N = 10240, K = 3072 9.3 -> 8.7; N = 12288, K = 4096 11.5 -> 9.8).
//   Five and more, q4f16_1, up to 8 rows from K = 3840 on (M = 8, N = 27648 19.0 -> 17.0, K = 4096 18.3 -> 17.2; K = 3584, N = 22016
//     13.3 -> 14.5); with 9 .. 16 rows, both formats, above 3072 (M = 9 / 16, N = 22016, K = 4096 18.8 / 19.5 -> 16.1 / 17.5 and
//     18.9 / 20.7 -> 16.4 / 18.0; q4f16_1 N = 49152, K = 3072 26.5 / 27.7 -> 27.3 / 28.3).
//   9 .. 16 rows, more than two, AutoGPTQ, where at least 15/16 of the pieces are K (M = 9 / 16, N = 12288, K = 4096 12.6 / 13.4 ->
//     10.5 / 11.9; with less than that N = 14336, K = 6400 17.3 / 19.8 -> 18.4 / 20.6).  q4f16_1 is as fast either way.
inline bool held_pays(HeldFormat fmt, int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = (N + 15) / 16, cus = cu_count();
  if (K > 4096 && tiles >= 4 * cus) return true;
  if (M <= 8) return (tiles > 2 * cus && K >= (fmt == kHeldGptq ? 3072 : 4352)) || (tiles >= 5 * cus && K >= 3840);
  if (tiles >= 5 * cus && K > 3072) return true;
  return fmt == kHeldGptq && tiles > 2 * cus && K > 3840 && 16 * K > 15 * 2048 * (int64_t)held_pieces(K);
}

// the kernel of a call: by that rule, or as the overrides for tests and measurement say (tuning.h; waves 2: activations in
// registers wherever they fit)
inline bool held_takes(HeldFormat fmt, int64_t M, int64_t N, int64_t K) {
  const Tuning& t = tuning();
  if (!held_fits(M, N, K)) return false;
  return t.skinny_waves == 2 || (!t.skinny_waves && !t.skinny_nw && !t.skinny_stages && held_pays(fmt, M, N, K));
}

template <HeldFormat FMT, int MODE, int PW, class Epilogue>
static int launch_held_form(const char* who, const HeldArgs& args, const uint16_t* x, uint16_t* y, const Epilogue& epi,
                            int64_t M, int64_t N, int64_t K, hipStream_t stream) {
  using Cfg = HeldCfg<FMT, MODE, PW>;
  auto kern = held_gemm_kernel<FMT, MODE, PW, Epilogue>;
  const int64_t tiles = (N + 15) / 16, rounds = (tiles + cu_count() - 1) / cu_count();
  static DynamicLdsLimit limit;  // per instantiation
  WQ_HIP(limit.ensure(reinterpret_cast<const void*>(kern), Cfg::kLdsBytes));
  // (as few workgroups as make the same number of rounds: each of them loads all activations)
  WQ_LAUNCH(who, kern, dim3((unsigned)((tiles + rounds - 1) / rounds)), dim3(512), Cfg::kLdsBytes, stream, args, (const half_t*)x,
            (half_t*)y, epi, (int)M, (int)N, (int)K);
  tuning().small_batch_form = kHeldForm;
  return WQ_OK;
}

template <HeldFormat FMT, class Epilogue>
static int launch_held(const char* who, const HeldArgs& args, const uint16_t* x, uint16_t* y, const Epilogue& epi, int64_t M,
                       int64_t N, int64_t K, hipStream_t stream) {
#define WQ_HELD_GO(MODE, PW) \
  if (held_pieces(K) == PW) return launch_held_form<FMT, MODE, PW, Epilogue>(who, args, x, y, epi, M, N, K, stream)
  if (M <= 8) {
    WQ_HELD_GO(0, 1);
    WQ_HELD_GO(0, 2);
    WQ_HELD_GO(0, 3);
    WQ_HELD_GO(0, 4);
    WQ_HELD_GO(0, 5);
  } else {
    WQ_HELD_GO(1, 1);
    WQ_HELD_GO(1, 2);
    WQ_HELD_GO(1, 3);
    WQ_HELD_GO(1, 4);
  }
#undef WQ_HELD_GO
  return fail(WQ_EINVAL, "%s: internal: M=%lld, K=%lld do not fit", who, (long long)M, (long long)K);
}

}  // namespace wq
#endif  // RELAX_AMD_CSRC_HELD_GEMM_H_
