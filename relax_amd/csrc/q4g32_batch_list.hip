// A list of format-A (q4f16_1) linears with 2 .. 32 activation rows each, in ONE launch.
//
// The counterpart of q4g32_gemv_list.hip for a small batch: the same persistent grid (one workgroup
// per CU walks the list, device-side counters order dependent linears), but the products are done by
// the matrix cores so that all M rows share one pass over the weights, and the weights go from
// memory straight into the registers that feed them.
//
// Two kernels: up to 16 rows of activations the one described here (q4g32_batch_list_kernel), beyond that
// q4g32_batch_rows_kernel further down, which shares the unpack, the lane exchange and the staging of activations.
//
// Work.  The unit is a TILE of rows of W times a PANEL of K: RT row tiles (1 or 2, 16 rows each) x 2048 or 4096 k (SP = 1 or
// 2).  A linear is run by one GROUP of workgroups (see batch_assign_groups), its tiles dealt to them round-robin, with a
// rotation that continues from linear to linear.  Inside a workgroup the 8 compute wavefronts split the panel 8 ways along
// K, each for all rows of the item.  A load is 8 rows x 128 bytes, 16 a lane; a lane's 16 bytes are the 32 codes of a scale
// group.
//
// Products.  What bounds this kernel is the vector unit beside the memory: with (q - 7) * s made in packed fp16, 13
// instructions per 8 weights and lane at 4 cycles a wavefront, it was busy for more than half of the launch.  (Measured per
// SIMD with two or more wavefronts: and, shift, add and fma of registers or literals take 2 cycles, packed and three-operand
// bit instructions 4, lane swaps 8.)  So a weight is not made at all.  A word's codes become fp16 numbers by masks alone (4
// ands and a shift): the code in bits 0 .. 3 of a half is the number 2^-24 q, in bits 4 .. 7 2^-20 q, and the activations of
// the former are taken 16 times when they are staged.  One v_mfma_f32_16x16x32_f16 takes the 32 codes of ONE group of 16
// rows, beginning at -7 times the group's sum of activations (another such product, with -7 in the codes' place), and 4
// fmas add the scale times that to the sums in fp32.  For one product to hold one group, the words of a group lie in
// the four lane quarters: two lane swaps for two words.  Nothing is rounded before the sums, in which the matrix core aligns
// products to 2^-17 of the largest: against 64 bits the error is that of the fp16 output (2.08e-4, of which its rounding is
// 2.07e-4; with rounded weights 2.74e-4), for activations of 1e-4 too (divided by 16 in the other positions 2.0e-3).
//   Up to 8 activation rows the 16 rows of the operand hold each of them twice, at the groups of the two halves of a
// 128-byte piece, so that lanes (rows, half) of a load are columns of one product as they come: half of the results, row
// half against other column half, are sums of nothing and are dropped.  With 9 .. 16 rows (WIDE) two loads exchange halves
// first (2 DPP moves a word more).
//   7 times an infinite sum is not what the products would give without it, so activations that are infinite or not a number
// take weights as the format defines them; so do linears of fewer rows than a row tile, whose few outputs may all be
// small, which is where the two roundings show.
// 32 layers of Llama-2-7B, M = 2 / 8 / 16: 774 / 762 / 785 -> 654 / 690 / 790 us (unpack as above; WIDE gains where lists are
// short: one layer, M = 16, 78 -> 52 us, hidden 8192, ffn 28672, 3 layers 582 -> 411).
//
// The other four wavefronts keep everything irregular away from that loop, through LDS:
//   * 2 x wavefronts wait for a producer linear (bounded spin), load a panel of activations,
//     rearrange it and leave it in one of 1 or 2 LDS buffers (under load a round trip to L2 takes several
//     microseconds); the compute wavefronts copy their slice into registers when they reach the panel,
//     which frees the buffer at once, so even one buffer keeps the next panel ready in time.  The two take
//     whole panels by turns: while one waits for a producer the other already fetches the panel after it
//     (sharing every panel between them instead was slower at every M).
//   * the scale wavefront streams the tile's scales (per row up to 256 contiguous bytes: fetched per
//     lane they cost more than the codes) into a ring of LDS slots, a few tiles ahead.
//   * the y wavefront adds the 8 partial sums of a tile in a fixed order, keeps the
//     sum in LDS while further panels of the same rows follow, and at the last panel applies bias / cast / residual,
//     stores y with device-scope stores and signals the linear's completion counter.
// A linear of several panels whose kept sums would not fit the LDS is walked in CHUNKS of its tiles (all
// panels of a chunk, then the next chunk; template parameter CH): the activations are then loaded once
// per chunk, which the host weighs against fewer, larger groups when it plans the list.
// Codes in flight: an item per wavefront, each load of which is replaced by the next item's as soon as its registers have
// been read (8 wavefronts x 8 KiB; 16 KiB per CU in flight reach the rate of the memory, 32 all of it).
#include <algorithm>
#include <cmath>
#include <vector>

#include "code_products.h"
#include "gemv_list_common.h"
#include "tuning.h"

namespace wq {

constexpr int kBW = 8;     // compute wavefronts: K slices of a panel
constexpr int kBXW = 2;    // wavefronts that stage activations
constexpr int kBRing = 4;  // LDS slots of scales and of partial sums: how far the compute wavefronts may spread
constexpr int kBThreads = 64 * (kBW + kBXW + 2);

// LDS words that hand the buffers over inside a workgroup (items = (linear, panel, tile) in the
// order the workgroup walks them; panels counted over all linears)
constexpr int kBMaxXBuf = 2;
constexpr int kBOddRows = 8;  // panels of which odd_rows is kept: the y wavefront is at most ring + kBMaxXBuf <= 6 behind the one staged
struct BatchFlags {
  int x_ready[kBMaxXBuf];  // [panel mod buffers] = panel + 1 once that panel's activations are staged
  int x_taken[kBMaxXBuf];  // [panel mod buffers] += 1 by each compute wavefront that has copied the panel
                           // (per buffer: with two buffers a wavefront may be a panel ahead of another)
  int s_ready;       // items whose scales are staged
  int y_done;        // items whose partial sums have been added up
  int abort;         // a wait of this workgroup ran into the spin limit: nobody waits any more
  int pad;
  int done[kBRing];  // += 1 by each compute wavefront per item finished, by slot (item mod ring)
  uint16_t odd_rows[kBOddRows];  // [panel mod kBOddRows]: rows of activations staged a sixteenth as large as the others
};
static_assert(sizeof(BatchFlags) == 64, "flags layout");

// Waits inside a workgroup are bounded like the waits between workgroups: a hand-over that never comes
// (a defect, or a wavefront that died) ends as an error word and a launch that finishes, not as a hang.
struct BatchWait {
  BatchFlags* flags;
  int* error;  // the list's error word
  long long limit;
  __device__ __forceinline__ void until(const int* flag, int target, int code) const {
    if (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >= target) {
      asm volatile("" ::: "memory");
      return;
    }
    const long long t0 = wall_clock64();
    while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < target) {
      if (__hip_atomic_load(&flags->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) break;
      if (wall_clock64() - t0 > limit) {
        __hip_atomic_store(&flags->abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __hip_atomic_store(error, kBatchInternalWait + code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    asm volatile("" ::: "memory");  // LDS is served in order: what was written before the flag is visible now
  }
};

// WIDE: 9 .. 16 activation rows (else up to 8); RT: row tiles (16 rows of W) per item; SP: the 8 compute wavefronts split a
// panel 8 ways along K, SP 128-byte pieces of every row of the item each.
__host__ __device__ constexpr int batch_panel_groups(int SP) { return kBW * 8 * SP; }
__host__ __device__ constexpr int batch_scale_row_bytes(int SP) { return batch_panel_groups(SP) * 2 + 16; }  // + 16: rows on different banks
__host__ __device__ constexpr int batch_scale_slot_bytes(int SP, int RT) { return 16 * RT * batch_scale_row_bytes(SP); }
__host__ __device__ constexpr int batch_partial_bytes(bool wide) { return wide ? 1024 : 512; }  // of a wavefront and row tile: 8 or 16 activation rows
__host__ __device__ constexpr int batch_partial_slot_bytes(bool wide, int RT) { return kBW * RT * batch_partial_bytes(wide); }
__host__ __device__ constexpr int batch_kept_bytes(int RT) { return RT * 1024; }  // sums of a tile kept between panels

// ---- the walk of a workgroup over its items.  All fields are wavefront-uniform.
struct ItemCursor {
  int lin;           // current linear (nlin: past the end)
  int panel, lt;     // panel of K, local tile (tile = lt * ncu + rb)
  int lt0, ltend;    // the current chunk of local tiles: a linear of several panels is walked chunk by chunk, all
                     // panels of a chunk before the next chunk, so that LDS holds the sums of one chunk only
  int csize;         // tiles per chunk of this linear
  int T, P;          // tiles of this workgroup in the linear (> 0), panels
  int ncu, rb;       // workgroups in the linear's group; (member - off) mod ncu
  int N, G, row_w;   // rows, scale groups per row, bytes per row of W
  const char* W;
  const char* S;
};

// word 16 of a descriptor: gmod_log2 | gidx << 8 | rows << 16 (read as one word: a scalar load; single
// bytes would come through a vector load and end up in vector registers)
// Which workgroups run a linear (bits 0 .. 15 of that word), in two forms:
//   * gmod_log2 = g < 0x80: the workgroups with b mod 2^g == gidx (for g = 3 one XCD: workgroup b runs on XCD
//     b mod 8, so the activations stay in that XCD's L2);
//   * gmod_log2 = 0x80: gidx is a MASK of XCDs, the group is every workgroup whose b mod 8 is in the mask.  This is
//     what a short list uses: its few linears share the 8 XCDs in proportion to their bytes.
// A member's index counts the members in order of b.
struct GroupOf {
  bool member;
  int index, size;
};
__device__ __forceinline__ int group_size(uint32_t grp, int nwg) {
  if (grp & 0x80u) return (nwg >> 3) * __builtin_popcount((grp >> 8) & 0xffu);
  return nwg >> (grp & 0x7fu);
}
__device__ __forceinline__ GroupOf group_of(uint32_t grp, int b, int nwg) {
  GroupOf r;
  if (grp & 0x80u) {
    const uint32_t mask = (grp >> 8) & 0xffu;
    const int pc = __builtin_popcount(mask);
    r.member = (mask >> (b & 7)) & 1u;
    r.index = (b >> 3) * pc + __builtin_popcount(mask & ((1u << (b & 7)) - 1u));
    r.size = (nwg >> 3) * pc;
  } else {
    const int gl = (int)(grp & 0x7fu);
    r.member = (b & ((1 << gl) - 1)) == (int)((grp >> 8) & 0xffu);
    r.index = b >> gl;
    r.size = nwg >> gl;
  }
  return r;
}

__device__ __forceinline__ uint32_t desc_group_word(gemv_desc_ptr descs, int lin) {
  typedef const uint32_t __attribute__((address_space(4)))* words_ptr;
  return ((words_ptr)(descs + lin))[16];
}

// positions the cursor on the first linear >= c.lin in which this workgroup holds a tile
template <int PG, bool CH>
__device__ __forceinline__ void item_seek(ItemCursor& c, gemv_desc_ptr descs, int nlin, int b, int nwg, int chunk) {
  typedef const uint32_t __attribute__((address_space(4)))* words_ptr;
  while (c.lin < nlin) {
    const words_ptr p = (words_ptr)(descs + c.lin);
    const uint32_t grp = p[16];
    const GroupOf go = group_of(grp, b, nwg);
    if (go.member) {  // this workgroup's group runs the linear
      uint32_t w[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) w[i] = p[i];
      const int ncu = go.size;
      int rb = go.index - (int)(w[15] >> 16);
      if (rb < 0) rb += ncu;
      const int T = (int)w[13] + (rb < (int)(w[15] & 0xffffu) ? 1 : 0);
      if (T > 0) {
        const int G = (int)(w[14] & 0xffffu);
        c.T = T;
        c.rb = rb;
        c.ncu = ncu;
        c.G = G;
        c.P = (G + PG - 1) / PG;
        c.N = (int)w[12];
        c.row_w = G << 4;
        c.W = reinterpret_cast<const char*>(((uint64_t)w[1] << 32) | w[0]);
        c.S = reinterpret_cast<const char*>(((uint64_t)w[3] << 32) | w[2]);
        c.panel = 0;
        c.lt = 0;
        if constexpr (CH) {
          c.lt0 = 0;
          // chunks of equal size, at most `chunk` tiles (one panel: no sums are kept, one chunk)
          c.csize = T;
          if (c.P > 1 && T > chunk) {
            const int nch = (T + chunk - 1) / chunk;
            c.csize = (T + nch - 1) / nch;
          }
          c.ltend = c.csize;
        }
        return;
      }
    }
    ++c.lin;
  }
}

template <int PG, bool CH>
__device__ __forceinline__ void item_next_panel(ItemCursor& c, gemv_desc_ptr descs, int nlin, int b, int nwg, int chunk) {
  if constexpr (CH) {
    if (++c.panel == c.P) {
      c.panel = 0;
      c.lt0 = c.ltend;
      if (c.lt0 >= c.T) {
        ++c.lin;
        item_seek<PG, CH>(c, descs, nlin, b, nwg, chunk);
        return;
      }
      c.ltend = min(c.T, c.lt0 + c.csize);
    }
    c.lt = c.lt0;
  } else {
    c.lt = 0;
    if (++c.panel == c.P) {
      ++c.lin;
      item_seek<PG, CH>(c, descs, nlin, b, nwg, chunk);
    }
  }
}

template <int PG, bool CH>
__device__ __forceinline__ void item_next(ItemCursor& c, gemv_desc_ptr descs, int nlin, int b, int nwg, int chunk) {
  if (++c.lt == (CH ? c.ltend : c.T)) item_next_panel<PG, CH>(c, descs, nlin, b, nwg, chunk);
}

template <bool WIDE, int SP, int RT, bool CH>
__global__ __launch_bounds__(kBThreads) void q4g32_batch_list_kernel(const GemvListDesc* __restrict__ descs_, int nlin,
                                                                     int* __restrict__ sync, long long spin_limit,
                                                                     int M, int nxb, int ring, int chunk, int use_sync) {
  constexpr int SG = 8 * SP, PG = batch_panel_groups(SP);  // scale groups per wavefront, and per panel
  constexpr int XO = WIDE ? 2 * SP : SP;  // sets of four operands that hold a wavefront's activations
  constexpr int NL = 2 * RT * SP;       // loads per wavefront and item, 8 rows x 128 bytes each
  constexpr int SROW = batch_scale_row_bytes(SP), SSLOT = batch_scale_slot_bytes(SP, RT);
  extern __shared__ uint4_t smem[];
  const gemv_desc_ptr descs = (gemv_desc_ptr)descs_;
  char* lds = reinterpret_cast<char*>(smem);
  // flags | nxb panels of activations, M x PG x 64 bytes each | `ring` scale slots | `ring` partial-sum slots |
  // sums kept between panels.  `ring` (2 or 4) is how many items the compute wavefronts may spread over.
  BatchFlags* flags = reinterpret_cast<BatchFlags*>(lds);
  char* const xbuf = lds + sizeof(BatchFlags);
  const int xbuf_bytes = M * (PG * 64);
  char* const sbuf = xbuf + nxb * xbuf_bytes;
  char* const pbuf = sbuf + ring * SSLOT;
  char* const abuf = pbuf + ring * batch_partial_slot_bytes(WIDE, RT);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nwg = gridDim.x;
  const int b = blockIdx.x;
  const BatchWait wait{flags, sync + sync_error_index(nlin), spin_limit > 0 ? spin_limit : 1000000};

  if (tid < (int)(sizeof(BatchFlags) / sizeof(int))) reinterpret_cast<int*>(flags)[tid] = 0;
  lds_done_then_barrier();  // LDS starts undefined: the flags are cleared before anyone looks

  if (wave < kBW) {
    // =========================== compute wavefront ===========================
    const int i = lane & 15, kq = lane >> 4;
    const int ks = wave;  // K slice of the panel
    // What has been requested: the item that is multiplied next, each load of which is replaced by that of the item behind it
    // as soon as its contents have been taken.  Past the last item the loads are issued too, against a descriptor that
    // holds nothing: without a branch around them the compiler counts how many are younger than the one it waits for.
    uint4_t buf[NL];
    ItemCursor ic, cc;
    ic.lin = 0;
    item_seek<PG, CH>(ic, descs, nlin, b, nwg, chunk);
    int k = 0;    // items consumed
    int pk = -1;  // panels taken
    // The activations of the slice as A operands.  Up to 8 rows: lane (i, kq) holds row i mod 8 at the groups of the half
    // i / 8 of a 128-byte piece, so that one operand serves what both halves of the lanes have loaded.
    half8_t xb[XO][4];
    bool special = false;
    const int xrows16 = WIDE ? M : 2 * M;
    const int xrow = WIDE ? min(i, M - 1) : (i >> 3) * M + min(i & 7, M - 1);
    const half8_t seven = __builtin_bit_cast(half8_t, uint4_t{0x80078007u, 0x80708070u, 0x80078007u, 0x80708070u});
    auto sevenfold = [&](int v, int g) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(xb[v][g], seven, float4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0); };

    struct Place {
      wq_rsrc_t base;
      uint32_t roff[2 * RT], goff[SP];
    };
    auto place_of = [&](const ItemCursor& c) {
      Place p;
      const int n0 = (c.lt * c.ncu + c.rb) * (16 * RT);
      const int rows = min(16 * RT, c.N - n0);           // >= 1
      const int pg = min(PG, c.G - c.panel * PG);        // scale groups of this panel (the last may be short)
      const uint64_t at = (uint64_t)(c.W + (int64_t)n0 * c.row_w + c.panel * (PG * 16));
      p.base = wq_rsrc((const char*)at, wq_live(c.lin, nlin));
      // Whole 128-byte lines: a load takes 8 rows, lane (i, kq) the 16 bytes of group 4 (i / 8) + kq of row i mod 8 (16 rows x
      // 64 bytes an instruction stream slower: 5.7 against 7.1 TB/s on 1 GiB with unpack and MFMAs).
      // Rows past N repeat the last row (never stored); groups past K repeat the last group (their
      // activations and scales are staged as zeros).
#pragma unroll
      for (int sp = 0; sp < SP; ++sp) p.goff[sp] = (uint32_t)min(ks * SG + (i >> 3) * 4 + kq + 8 * sp, pg - 1) * 16u;
#pragma unroll
      for (int r = 0; r < 2 * RT; ++r) p.roff[r] = __umul24((uint32_t)min(8 * r + (i & 7), rows - 1), (uint32_t)c.row_w);
      return p;
    };
    auto request = [&](const Place& p, int sp, int r) { return __builtin_amdgcn_raw_buffer_load_b128(p.base, p.roff[r] + p.goff[sp], 0, kNonTemporal); };

    // 8 codes as the weights that the format defines, (q - 7) * s rounded to fp16, times 16 in bits 4 .. 7
    auto weights = [&](uint32_t w, half_t s) {
      const half2_t c7 = {(half_t)-1031.0f, (half_t)-1031.0f}, c112 = {(half_t)-1136.0f, (half_t)-1136.0f}, s2 = {s, s};
      const uint4_t c = __builtin_bit_cast(uint4_t, code_operand(w)) | 0x64006400u;
      return __builtin_bit_cast(half8_t, uint4_t{as_u32((as_half2(c.x) + c7) * s2), as_u32((as_half2(c.y) + c112) * s2),
                                                 as_u32((as_half2(c.z) + c7) * s2), as_u32((as_half2(c.w) + c112) * s2)});
    };
    // the lane's four scales of what load r of piece sp brought (WIDE: of chunk r mod 2 of row tile r / 2)
    auto scales = [&](int slot, int sp, int r) {
      const int row = WIDE ? (r >> 1) * 16 + i : 8 * r + (i & 7), group = ks * SG + 8 * sp + 4 * (WIDE ? r & 1 : i >> 3);
      return *reinterpret_cast<const half4_t*>(sbuf + slot * SSLOT + row * SROW + group * 2);
    };

    constexpr int NA = WIDE ? RT : 2 * RT;  // accumulators: row tiles, or halves of row tiles
    constexpr int QB = RT < 2 ? RT : 2;     // row tiles at a time
    auto multiply = [&](const Place& next, int slot, float4_t (&acc)[NA]) {
#pragma unroll
      for (int blk = 0; blk < SP * (RT / QB); ++blk) {
        const int sp = blk / (RT / QB), q0 = blk % (RT / QB) * QB;
        uint32_t w[2 * QB][4];
        half4_t s4[2 * QB];
        // in steps of two products, and behind them the scaling of those of the step before
        float4_t t[2][2], c[WIDE ? 2 : 1];
        auto scale = [&](int step) {
          const int g = step / QB, q = step % QB;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            float4_t& a = acc[WIDE ? q0 + q : 2 * (q0 + q) + h];
#pragma unroll
            for (int e = 0; e < 4; ++e) a[e] = fmaf(t[step & 1][h][e], (float)s4[2 * q + h][g], a[e]);
          }
        };
#pragma unroll
        for (int step = 0; step < 4 * QB; ++step) {
          const int g = step / QB, q = step % QB;
          if (g == 0) {
#pragma unroll
            for (int r = 2 * q; r < 2 * q + 2; ++r) {
              const int at = sp * 2 * RT + 2 * q0 + r;
              take_words(buf[at], w[r]);
              buf[at] = request(next, sp, 2 * q0 + r);
              s4[r] = scales(slot, sp, 2 * q0 + r);
            }
            if constexpr (WIDE) exchange_halves(w[2 * q], w[2 * q + 1]);
            spread_words(w[2 * q]);
            spread_words(w[2 * q + 1]);
          }
          if (q == 0) {
#pragma unroll
            for (int v = 0; v < (WIDE ? 2 : 1); ++v) c[v] = sevenfold(WIDE ? 2 * sp + v : sp, g);
          }
#pragma unroll
          for (int h = 0; h < 2; ++h)
            t[step & 1][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xb[WIDE ? 2 * sp + h : sp][g], code_operand(w[2 * q + h][g]), c[WIDE ? h : 0], 0, 0, 0);
          if (step > 0) scale(step - 1);
          __builtin_amdgcn_sched_barrier(0);
        }
        scale(4 * QB - 1);
      }
    };
    // The same with rounded weights, straight from memory: for activations that are infinite or not a number (7 times one
    // of those is not what the sum of the products would be without it), and for fewer rows than a row tile.
    auto multiply_rounded = [&](const Place& next, int slot, float4_t (&acc)[NA]) {
      const Place here = place_of(cc);
#pragma unroll
      for (int sp = 0; sp < SP; ++sp)
#pragma unroll
        for (int q = 0; q < RT; ++q) {
          uint32_t w[2][4];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const uint4_t l = request(here, sp, 2 * q + h);
            w[h][0] = l.x, w[h][1] = l.y, w[h][2] = l.z, w[h][3] = l.w;
          }
          if constexpr (WIDE) exchange_halves(w[0], w[1]);
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            spread_words(w[h]);
            const half4_t s4 = scales(slot, sp, 2 * q + h);
            float4_t& a = acc[WIDE ? q : 2 * q + h];
#pragma unroll
            for (int g = 0; g < 4; ++g) a = __builtin_amdgcn_mfma_f32_16x16x32_f16(xb[WIDE ? 2 * sp + h : sp][g], weights(w[h][g], s4[g]), a, 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
      for (int q = 0; q < NA; ++q) acc[q] *= 1.0f / 16777216.0f;  // (like the products of codes, 2^-20 of the weights' of x)
#pragma unroll
      for (int sp = 0; sp < SP; ++sp)
#pragma unroll
        for (int r = 0; r < 2 * RT; ++r) {
          buf[sp * 2 * RT + r] = request(next, sp, r);
          __builtin_amdgcn_sched_barrier(0);  // in this order everywhere: the waits count on it
        }
    };

    auto consume = [&](const Place& next) {
      if (cc.lt == (CH ? cc.lt0 : 0)) {
        // a new panel: its activations are staged (or will be); this wavefront's K slice goes to registers
        ++pk;
        const int xslot = pk % nxb;
        wait.until(&flags->x_ready[xslot], pk + 1, 1);
        const char* xs = xbuf + xslot * xbuf_bytes + ((ks * (XO * 16) + kq) * xrows16 + xrow) * 16;
#pragma unroll
        for (int v = 0; v < XO; ++v)
#pragma unroll
          for (int g = 0; g < 4; ++g) xb[v][g] = *reinterpret_cast<const half8_t*>(xs + ((v * 4 + g) * 4 * xrows16) * 16);
        float zero = 0.0f;  // NaN where an activation is infinite or not a number
#pragma unroll
        for (int v = 0; v < XO; ++v)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const float4_t c = sevenfold(v, g);
#pragma unroll
            for (int e = 0; e < 4; ++e) zero = fmaf(c[e], 0.0f, zero);
          }
        special = __builtin_amdgcn_ballot_w64(zero != 0.0f) != 0;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (lane == 0) __hip_atomic_fetch_add(&flags->x_taken[xslot], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      wait.until(&flags->s_ready, k + 1, 2);
      const int slot = k & (ring - 1);
      float4_t acc[NA];
#pragma unroll
      for (int q = 0; q < NA; ++q) acc[q] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
      if (special || cc.N < 16) multiply_rounded(next, slot, acc);
      else multiply(next, slot, acc);
      if (k >= ring) wait.until(&flags->y_done, k - ring + 1, 3);
      // sums as [row tile][activation row][row of W]
      float* const part = reinterpret_cast<float*>(pbuf + (slot * kBW + wave) * (RT * batch_partial_bytes(WIDE)));
#pragma unroll
      for (int q = 0; q < RT; ++q) {
        if constexpr (!WIDE) {
          float sum[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[e] = join_halves(acc[2 * q][e], acc[2 * q + 1][e]);
          if (i < 8) {
#pragma unroll
            for (int e = 0; e < 4; ++e) part[q * 128 + (4 * (kq & 1) + e) * 16 + 8 * (kq >> 1) + i] = sum[e];
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) part[q * 256 + (4 * kq + e) * 16 + i] = acc[q][e];
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (lane == 0) __hip_atomic_fetch_add(&flags->done[slot], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      ++k;
    };

    if (ic.lin >= nlin) return;
    {
      const Place p = place_of(ic);
#pragma unroll
      for (int sp = 0; sp < SP; ++sp)
#pragma unroll
        for (int r = 0; r < 2 * RT; ++r) {
          buf[sp * 2 * RT + r] = request(p, sp, r);
          __builtin_amdgcn_sched_barrier(0);
        }
    }
    while (ic.lin < nlin) {
      cc = ic;
      item_next<PG, CH>(ic, descs, nlin, b, nwg, chunk);
      consume(place_of(ic));
    }
    return;
  }

  bool aborted = false;

  if (wave < kBW + kBXW) {
    // ====================== x wavefronts: a panel of activations -> LDS ======================
    const int xw = wave - kBW;
    // until every workgroup has signalled linear `dep`, or the spin limit passes
    auto wait_for = [&](int dep) {
      if (aborted) return;
      const long long t0 = wall_clock64();
      while (true) {
        // read-modify-write (+ 0): performed where the counter lives, never served from a stale cache line
        int v = 0;
        if (lane < kCountersPerLinear)
          v = __hip_atomic_fetch_add(sync + sync_counter_index(dep, lane), 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        v += __shfl_xor(v, 1, 64);
        v += __shfl_xor(v, 2, 64);
        v += __shfl_xor(v, 4, 64);
        if (__builtin_amdgcn_readfirstlane(v) >= group_size(desc_group_word(descs, dep), nwg)) break;  // every member of its group
        if (wall_clock64() - t0 > spin_limit) {
          aborted = true;
          if (lane == 0)
            __hip_atomic_store(sync + sync_error_index(nlin), dep + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
        __builtin_amdgcn_s_sleep(4);
      }
      // whatever this XCD's L2 still holds of an earlier content of x (the addresses are reused
      // from launch to launch) must not serve the loads that follow
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    };

    // A code in bits 0 .. 3 of a half counts a sixteenth of one in bits 4 .. 7: the activations of the former are staged 16
    // times.  (Those of the latter divided by 16 lose bits below 2^-10.)  A row of the panel in which that gives an
    // infinity, where an activation is 4096 or more, is staged once and a sixteenth, and its sums are taken 16 times: what
    // that costs, 2^-21 of an activation, is nothing beside the large one, and no other row changes.
    const half2_t sixteen = {(half_t)16.0f, (half_t)16.0f}, sixteenth = {(half_t)0.0625f, (half_t)0.0625f}, one = {(half_t)1.0f, (half_t)1.0f}, null2 = {(half_t)0.0f, (half_t)0.0f};
    constexpr int PPR = PG * 4;  // 16-byte pieces (8 activations) per row and panel; a power of two
    constexpr int UX = 32;       // loads in flight per lane: one round trip for a panel of 8 rows x 2048 k
    constexpr int UR = PPR / 64; // loads of a row
    static_assert(UX % UR == 0, "whole rows are loaded");
    const int xrows16 = WIDE ? M : 2 * M;
    // 64 pieces are 16 groups of a row, four dwords each: one slice, or two (WIDE).  The order is that of the operands.
    const int c = lane >> 2, d = lane & 3;
    const int place0 = WIDE ? c : (c >> 3) * 4 + (c & 3), half = WIDE ? 0 : (c >> 2) & 1;
    ItemCursor xc;
    xc.lin = 0;
    item_seek<PG, CH>(xc, descs, nlin, b, nwg, chunk);
    // the x wavefronts take whole panels by turns (panel pk belongs to wavefront pk mod kBXW) and run up
    // to nxb panels ahead of the compute wavefronts: under load a round trip to L2 takes several microseconds
    int pk = 0;
    int confirmed = -1;  // the latest producer linear this wavefront has seen complete
    while (xc.lin < nlin) {
      if (pk % kBXW == xw) {
        const int xslot = pk % nxb;
        // the buffer is free once every compute wavefront has copied the panel that used it before
        if (pk >= nxb) wait.until(&flags->x_taken[xslot], kBW * (pk / nxb), 4);
        const int j = xc.lin;
        const int dep = (int)((descs[j].g_dep >> 16) & 0x7fffu) - 1;
        if (dep >= 0 && dep != confirmed) {
          wait_for(dep);
          confirmed = dep;
        }
        const int K = xc.G << 5;
        const int K8 = K >> 3;
        const int xrows = (int)((desc_group_word(descs, j) >> 16) & 0xffu);
        // an x that other workgroups of this launch have written is read with device-scope loads (sc1)
        const __amdgpu_buffer_rsrc_t xr =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(descs[j].x), 0, xrows * K * 2, kBufferFlags);
        char* const xdst = xbuf + xslot * xbuf_bytes;
        const int total = M * PPR;
        auto stage = [&](uint4_t v, int row, int t, half2_t low, half2_t high, float zero) {
          const uint32_t in[4] = {v.x, v.y, v.z, v.w};
          uint32_t p[4];
          pair_i_i4(in, p);  // p[e] = (x_e, x_{e+4})
          const half2_t p0 = as_half2(p[0]) * low, p2 = as_half2(p[2]) * low;
          const int first = t * (WIDE ? 16 : 8);
          *reinterpret_cast<uint4_t*>(xdst + (((first + place0) * 4 + d) * xrows16 + half * M + row) * 16) =
              uint4_t{as_u32(p0), as_u32(as_half2(p[1]) * high), as_u32(p2), as_u32(as_half2(p[3]) * high)};
          return dot2(p0, null2, dot2(p2, null2, zero));
        };
        uint32_t odd = 0;
        for (int base = 0; base < total; base += 64 * UX) {
          uint4_t v[UX];
#pragma unroll
          for (int t = 0; t < UX; ++t) {
            const int at = base + t * 64;  // (a row of a panel is whole wavefronts of pieces)
            const int go = xc.panel * PPR + (at & (PPR - 1));  // the place in the row of lane 0's piece
            const int src = min(at / PPR, xrows - 1);  // rows past the entry's repeat its last row (never stored)
            // Past the row, or the panel: an offset that the descriptor does not reach, which brings zeros.  The scalar offset of
            // such a load lies inside too, so that it does not matter whether the range check counts it (wq_device.h): it is 0
            // where no lane has a piece.
            const uint32_t off = at < total && go + lane < K8 ? (uint32_t)lane * 16u : 0x80000000u;
            const int start = (src * K8 + go) * 16 & wq_live(go, K8) & wq_live(at, total);
            v[t] = dep >= 0 ? __builtin_amdgcn_raw_buffer_load_b128(xr, off, start, kDeviceScope)
                            : __builtin_amdgcn_raw_buffer_load_b128(xr, off, start, 0);
          }
#pragma unroll
          for (int r = 0; r < UX / UR; ++r) {
            const int row = base / PPR + r;
            if (row < M) {
              float zero = 0.0f;  // NaN where 16 times an activation is infinite or not a number
#pragma unroll
              for (int t = 0; t < UR; ++t) zero = stage(v[r * UR + t], row, t, sixteen, one, zero);
              if (__builtin_amdgcn_ballot_w64(zero != 0.0f)) odd |= 1u << row;
            }
          }
        }
        for (uint32_t left = odd; left; left &= left - 1) {
          const int row = __builtin_ctz(left), src = min(row, xrows - 1);
#pragma unroll 1
          for (int t = 0; t < UR; ++t) {
            const int go = xc.panel * PPR + t * 64;
            const uint32_t off = go + lane < K8 ? (uint32_t)((src * K8 + go + lane) * 16) : 0x80000000u;
            stage(dep >= 0 ? __builtin_amdgcn_raw_buffer_load_b128(xr, off, 0, kDeviceScope) : __builtin_amdgcn_raw_buffer_load_b128(xr, off, 0, 0),
                  row, t, one, sixteenth, 0.0f);
          }
        }
        if (lane == 0) flags->odd_rows[pk % kBOddRows] = (uint16_t)odd;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (lane == 0) __hip_atomic_store(&flags->x_ready[xslot], pk + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      ++pk;
      item_next_panel<PG, CH>(xc, descs, nlin, b, nwg, chunk);
    }
    return;
  }

  if (wave == kBW + kBXW) {
    // ====================== scale wavefront: the scales of a tile -> LDS ======================
    constexpr int PD = NL <= 4 ? 6 : 3;  // items in flight in registers (a round trip under load is several items long)
    constexpr int PPR = PG / 8;      // 16-byte pieces (8 scales) per row and panel
    constexpr int LP = 16 * RT * PPR / 64;  // pieces per lane and item
    uint4_t sv[PD][LP];
    ItemCursor ic, cc;
    ic.lin = 0;
    item_seek<PG, CH>(ic, descs, nlin, b, nwg, chunk);
    cc = ic;
    int k = 0;
    auto issue = [&](uint4_t (&buf)[LP]) {
      if (ic.lin >= nlin) return;
      const int n0 = (ic.lt * ic.ncu + ic.rb) * (16 * RT);
      const int pg = min(PG, ic.G - ic.panel * PG);
      const char* base = ic.S + ic.panel * (PG * 2);
#pragma unroll
      for (int t = 0; t < LP; ++t) {
        const int idx = t * 64 + lane;
        const int r = idx / PPR, pc = idx % PPR;
        buf[t] = uint4_t{0, 0, 0, 0};  // groups past K: a zero scale
        if (pc * 8 < pg)
          buf[t] = __builtin_nontemporal_load(
              reinterpret_cast<const uint4_t*>(base + (int64_t)min(n0 + r, ic.N - 1) * (ic.G * 2) + pc * 16));
      }
      item_next<PG, CH>(ic, descs, nlin, b, nwg, chunk);
    };
    auto consume = [&](uint4_t (&buf)[LP]) {
      const int slot = k & (ring - 1);
      // the slot is free once every compute wavefront has finished the item that used it before
      if (k >= ring) wait.until(&flags->done[slot], kBW * (k / ring), 5);
#pragma unroll
      for (int t = 0; t < LP; ++t) {
        const int idx = t * 64 + lane;
        const int r = idx / PPR, pc = idx % PPR;
        *reinterpret_cast<uint4_t*>(sbuf + slot * SSLOT + r * SROW + pc * 16) = buf[t];
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      ++k;
      if (lane == 0) __hip_atomic_store(&flags->s_ready, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      item_next<PG, CH>(cc, descs, nlin, b, nwg, chunk);
    };
#pragma unroll
    for (int t = 0; t < PD - 1; ++t) issue(sv[t]);
    while (cc.lin < nlin) {
#pragma unroll
      for (int t = 0; t < PD; ++t) {
        issue(sv[(t + PD - 1) % PD]);
        if (cc.lin < nlin) consume(sv[t]);
      }
    }
    return;
  }

  // ================== y wavefront: partial sums -> y, completion signals ==================
  {
    const int j16 = lane & 15, rq = lane >> 4;
    int k = 0, pk = -1;
    for (int lin = 0; lin < nlin; ++lin) {
      const uint32_t g_dep = descs[lin].g_dep;
      const uint32_t grp = desc_group_word(descs, lin);
      const GroupOf go = group_of(grp, b, nwg);
      if (!go.member) continue;  // another group's linear
      const int ncu = go.size;
      int rb = go.index - (int)descs[lin].off;
      if (rb < 0) rb += ncu;
      const int T = descs[lin].q + (rb < (int)descs[lin].rem ? 1 : 0);
      const int N = descs[lin].N;
      const int P = ((int)(g_dep & 0xffffu) + PG - 1) / PG;
      int csize = T;
      if (CH && P > 1 && T > chunk) {
        const int nch = (T + chunk - 1) / chunk;
        csize = (T + nch - 1) / nch;
      }
      const half_t* bias = descs[lin].bias;
      const half_t* residual = descs[lin].residual;
      const int yrows = (int)((grp >> 16) & 0xffu);
      const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(descs[lin].y, 0, yrows * N * 2, kBufferFlags);
      // the four outputs of a lane are adjacent in a row of y: one 8-byte store where the addresses allow it
      // (a store instruction waits its turn behind the weight loads of the whole workgroup)
      const bool wide = (N & 3) == 0 && (((uintptr_t)descs[lin].y | (uintptr_t)bias | (uintptr_t)residual) & 7) == 0;
      for (int lt0 = 0; lt0 < T; lt0 += csize) {
        const int ltend = min(T, lt0 + csize);
        for (int panel = 0; panel < P; ++panel) {
          ++pk;
          for (int lt = lt0; lt < ltend; ++lt, ++k) {
            const int slot = k & (ring - 1);
            wait.until(&flags->done[slot], kBW * (k / ring + 1), 6);
            const float factor = (flags->odd_rows[pk % kBOddRows] >> j16) & 1 ? 16.0f : 1.0f;
            // sum[t]: rows 16 t + 4 rq .. + 3 of the tile, activation row j16; the K slices in a fixed order
            const char* pb = pbuf + slot * batch_partial_slot_bytes(WIDE, RT) + (WIDE ? j16 : j16 & 7) * 64 + rq * 16;
            float4_t sum[RT];
#pragma unroll
            for (int t = 0; t < RT; ++t) {
              sum[t] = *reinterpret_cast<const float4_t*>(pb + t * batch_partial_bytes(WIDE));
#pragma unroll
              for (int w = 1; w < kBW; ++w) sum[t] += *reinterpret_cast<const float4_t*>(pb + (w * RT + t) * batch_partial_bytes(WIDE));
            }
#pragma unroll
            for (int t = 0; t < RT; ++t) sum[t] *= factor;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (lane == 0) __hip_atomic_store(&flags->y_done, k + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (P > 1) {
              float4_t* keep = reinterpret_cast<float4_t*>(abuf + (lt - lt0) * batch_kept_bytes(RT) + lane * 16);
              if (panel > 0) {
#pragma unroll
                for (int t = 0; t < RT; ++t) sum[t] += keep[t * 64];
              }
              if (panel < P - 1) {
#pragma unroll
                for (int t = 0; t < RT; ++t) keep[t * 64] = sum[t];
                continue;
              }
            }
#pragma unroll
            for (int t = 0; t < RT; ++t) {
              // lane (j, rq) holds rows n0 + 4 rq .. + 3 of activation row j
              const int n0 = (((lt * ncu + rb) * RT + t) << 4) + 4 * rq;
              const float4_t v4 = sum[t] * 1048576.0f;  // (the products were 2^-20 of themselves)
              if (j16 < yrows && wide) {
                if (n0 < N) {
                  float4_t v = v4;
                  if (bias) {
                    const half4_t bv = *reinterpret_cast<const half4_t*>(bias + n0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] += (float)bv[e];
                  }
                  half4_t h = {(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
                  if (residual) h = h + *reinterpret_cast<const half4_t*>(residual + (int64_t)j16 * N + n0);
                  // device-scope store: written through, so that a counter update after it publishes it
                  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2_t, h), yr, (j16 * N + n0) * 2, 0, kDeviceScope);
                }
              } else if (j16 < yrows) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  const int n = n0 + e;
                  if (n < N) {
                    float v = v4[e];
                    if (bias) v += (float)bias[n];
                    half_t h = (half_t)v;
                    if (residual) h = h + residual[(int64_t)j16 * N + n];
                    __builtin_amdgcn_raw_buffer_store_b16(as_u16(h), yr, (j16 * N + n) * 2, 0, kDeviceScope);
                  }
                }
              }
            }
          }
        }
      }
      if (g_dep & kSignal) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stores of this workgroup have been written through
        if (lane == 0)
          __hip_atomic_fetch_add(sync + sync_counter_index(lin, b & (kCountersPerLinear - 1)), 1, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    if (!use_sync) return;
    // the last workgroup to get here clears the counters for the next launch (its own counter updates
    // have arrived by then: nothing of this launch may land on a cleared counter)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    int last = 0;
    if (lane == 0)
      last = __hip_atomic_fetch_add(sync + sync_finished_index(nlin), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
             nwg - 1;
    if (__builtin_amdgcn_readfirstlane(last)) {
      for (int i = lane; i < nlin * kCountersPerLinear; i += 64)
        __hip_atomic_store(sync + i * kCounterStride, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (lane == 0)
        __hip_atomic_store(sync + sync_finished_index(nlin), 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// ====================================================================================================
// More than 16 activation rows: the wavefront that owns rows of W keeps their sums.
//
// With 17 .. 32 rows of activations a panel of 1024 k fills 64 KiB of LDS, the kernel above then hands over
// items of 16 KiB, and what an item costs in hand-overs (partial sums through LDS, the y wavefront's
// epilogue, the sums kept between panels) is paid four times per 4096 k.  Here nothing is handed over but the
// operands: a compute wavefront owns up to TR = 4 ROW TILES (16 rows each) of W for ALL of K, its accumulators
// (TR x R x 4 registers) stay in registers from the first panel to the last, and it writes its own outputs.
// The 8 compute wavefronts of a workgroup walk the panels of activations together (a PASS of the workgroup:
// up to 8 x 64 rows; the activations are loaded once per pass, which is why TR is as large as the registers
// allow: 167 of the 168 that 11 wavefronts leave each other).
//   * The activations of a panel (512 k: M x 1 KiB) lie in LDS in B-operand order; every compute wavefront
//     reads the operand of a (step, dword) pair once and uses it for its TR row tiles (LDS reads: 2 bytes per
//     byte of codes).  Two x wavefronts stage panels by turns into `nxb` buffers; a buffer is free again when
//     all 8 compute wavefronts have left it.
//   * One scale wavefront stages the scales of the rows of a pass, 1024 k (64 bytes per row) at a time, into
//     2 buffers.
//   * The unit of the weight stream is a PAIR of chunks of a wavefront's rows: 256 k, per row tile two loads of
//     8 rows x 128 bytes (whole lines; a lane exchange puts the halves where the MFMA wants them), 2 TR loads
//     in all, waited for by hand.  A pair is first exchanged into registers of its own and its ring slot
//     refilled at once, so two pairs (32 KiB per wavefront) are in flight while one is multiplied.  The loads
//     are buffer loads on the wavefront's rows of the pass: past them (a short last pass, the end of W) a load brings
//     zeros or the first rows again, which are never stored; a wavefront without rows in a pass loads from
//     an empty buffer and only takes part in the hand-overs.
//   * A linear's completion counter is raised by the last of the 8 compute wavefronts to have its stores
//     written through.
// What bounds it (cycle counters around the phases of a compute wavefront, an instrumented copy): not memory.  A
// compute wavefront waits for its weights 1 % of the time; 43 .. 58 % goes into unpacking and multiplying a pair
// (about 1100 instructions, 6 .. 8 cycles each with two such wavefronts per SIMD), 13 .. 19 % into the lane
// exchange and the refill, and the wavefronts that share a SIMD with an older one are slower, so the older ones
// wait for them at the hand-over of the panels (35 % of their time).  Measured and not kept: B operands and
// scales requested from LDS one step ahead (no change), the refill spread over the multiplication (no change),
// a raised priority for the service wavefronts (M = 17 slower), 12 compute wavefronts of 48 rows (128 registers:
// 5 % slower), branches around the row tiles a short pass does not have (5 % slower: the unrolled code no longer
// interleaves).  The activations of every pass (M x K x 2 bytes per 512 rows: 22 % of the codes at M = 32)
// cost what their bytes cost: the stack step grows by 4.5 us per row of activations.
constexpr int kRW = 8;      // compute wavefronts
constexpr int kRXW = 2;     // wavefronts that stage activations
constexpr int kRThreads = 64 * (kRW + kRXW + 1);
constexpr int kRPairGroups = 8;   // scale groups per pair of chunks (256 k)
constexpr int kRPG = 16;          // scale groups per panel of activations
constexpr int kRSPG = 32;         // scale groups per panel of scales
constexpr int kRSRow = kRSPG * 2 + 16;  // LDS bytes per row of a panel of scales (+ 16: the 16 rows of a row tile on different banks)
constexpr int kRMaxXBuf = 4;

struct RowsFlags {
  int x_ready[kRMaxXBuf];  // [panel mod buffers] = panel + 1 once staged (panels counted over the whole launch)
  int x_taken[kRMaxXBuf];  // += 1 by each compute wavefront that has left the panel
  int s_ready[2], s_taken[2];  // the same for the panels of scales
  int lin_done[8];         // [linear mod 8] += 1 by each compute wavefront whose stores of the linear are written through
                           // (a wavefront is at most `nxb` <= 4 panels, hence linears, ahead of another)
  int exited;              // compute wavefronts that have finished the list
  int abort;               // a wait of this workgroup ran into the spin limit: nobody waits any more
  int pad[10];
};
static_assert(sizeof(RowsFlags) == 128, "flags layout");

struct RowsWait {
  int* abort;
  int* error;
  long long limit;
  __device__ __forceinline__ void until(const int* flag, int target, int code) const {
    if (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >= target) {
      asm volatile("" ::: "memory");
      return;
    }
    const long long t0 = wall_clock64();
    while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < target) {
      if (__hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) break;
      if (wall_clock64() - t0 > limit) {
        __hip_atomic_store(abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __hip_atomic_store(error, kBatchInternalWait + code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    asm volatile("" ::: "memory");
  }
};

// The walk of a workgroup over (linear, pass, pair of chunks).  All fields are wavefront-uniform.  A workgroup's
// share of a linear is a run of consecutive ROW TILES (16 rows); a pass takes up to 8 TR of them, `tr` per
// wavefront: TR while there are that many, and in the last pass as few as cover what is left with all 8
// wavefronts (three wave tiles of 64 rows left over: 6 wavefronts with 32 rows each, half the time).
struct RowsCursor {
  int lin;         // nlin: past the end
  int q, Q;        // pair of chunks within K
  int pos, left;   // first row tile of the pass; row tiles of the workgroup from there on (> 0)
  int tr;          // row tiles per wavefront in this pass (1 .. TR)
  int N, G, row_w;
  const char* W;
  const char* S;
  // row tiles of wavefront w in this pass, and the first of them
  __device__ __forceinline__ int tiles_of(int w, int TR) const { return max(0, min(tr, min(left, kRW * TR) - w * tr)); }
  __device__ __forceinline__ int first_of(int w) const { return pos + w * tr; }
};

template <int TR>
__device__ __forceinline__ void rows_begin_pass(RowsCursor& c) {
  c.q = 0;
  c.tr = (min(c.left, kRW * TR) + kRW - 1) / kRW;
}

// positions the cursor on the first linear >= c.lin in which this workgroup holds a row tile.  SIGNAL (the
// cursor that the first compute wavefront consumes with): a linear of this workgroup's group in which it
// holds none is signalled as complete on the way.
template <int TR, bool SIGNAL>
__device__ __forceinline__ void rows_seek(RowsCursor& c, gemv_desc_ptr descs, int nlin, int b, int nwg, int* sync, int lane) {
  typedef const uint32_t __attribute__((address_space(4)))* words_ptr;
  while (c.lin < nlin) {
    const words_ptr p = (words_ptr)(descs + c.lin);
    const uint32_t grp = p[16];
    const GroupOf go = group_of(grp, b, nwg);
    if (go.member) {  // this workgroup's group runs the linear
      const int ncu = go.size;
      const uint32_t w15 = p[15];
      int rb = go.index - (int)(w15 >> 16);
      if (rb < 0) rb += ncu;
      const int q = (int)p[13], rem = (int)(w15 & 0xffffu);
      const int cnt = q + (rb < rem ? 1 : 0);
      if (cnt > 0) {
        const uint32_t w14 = p[14];
        const int G = (int)(w14 & 0xffffu);
        c.left = cnt;
        c.pos = rb * q + min(rb, rem);
        c.G = G;
        c.Q = G / kRPairGroups;
        c.N = (int)p[12];
        c.row_w = G << 4;
        c.W = reinterpret_cast<const char*>(((uint64_t)p[1] << 32) | p[0]);
        c.S = reinterpret_cast<const char*>(((uint64_t)p[3] << 32) | p[2]);
        rows_begin_pass<TR>(c);
        return;
      }
      if (SIGNAL && (p[14] & kSignal) && lane == 0)
        __hip_atomic_fetch_add(sync + sync_counter_index(c.lin, b & (kCountersPerLinear - 1)), 1, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
    ++c.lin;
  }
}

template <int TR, bool SIGNAL>
__device__ __forceinline__ void rows_advance(RowsCursor& c, int step, gemv_desc_ptr descs, int nlin, int b, int nwg, int* sync, int lane) {
  c.q += step;
  if (c.q < c.Q) return;
  const int took = min(c.left, kRW * TR);
  c.pos += took;
  c.left -= took;
  if (c.left > 0) {
    rows_begin_pass<TR>(c);
    return;
  }
  ++c.lin;
  rows_seek<TR, SIGNAL>(c, descs, nlin, b, nwg, sync, lane);
}

template <int TR, int R>
__global__ __launch_bounds__(kRThreads) void q4g32_batch_rows_kernel(const GemvListDesc* __restrict__ descs_, int nlin,
                                                                     int* __restrict__ sync, long long spin_limit,
                                                                     int M, int nxb, int use_sync) {
  constexpr int TROWS = 16 * TR;                 // rows of a wave tile
  constexpr int SBUF = kRW * TROWS * kRSRow;     // bytes of a buffer of scales
  extern __shared__ uint4_t smem[];
  const gemv_desc_ptr descs = (gemv_desc_ptr)descs_;
  char* lds = reinterpret_cast<char*>(smem);
  // flags | nxb panels of activations, M x 1 KiB each | 2 panels of scales
  RowsFlags* flags = reinterpret_cast<RowsFlags*>(lds);
  char* const xbuf = lds + sizeof(RowsFlags);
  const int xbuf_bytes = M * (kRPG * 64);
  char* const sbuf = xbuf + nxb * xbuf_bytes;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nwg = gridDim.x;
  const int b = blockIdx.x;
  const RowsWait wait{&flags->abort, sync + sync_error_index(nlin), spin_limit > 0 ? spin_limit : 1000000};

  if (tid < (int)(sizeof(RowsFlags) / sizeof(int))) reinterpret_cast<int*>(flags)[tid] = 0;
  lds_done_then_barrier();

  if (wave < kRW) {
    // =========================== compute wavefront ===========================
    const int i = lane & 15, kq = lane >> 4;
    constexpr int NT = 2;        // ring slots: both in flight while a pair is multiplied (out of registers of its own)
    constexpr int LPI = 2 * TR;  // loads per pair
    // The ring is loaded in assembly and waited for by hand, as in the kernel above: `magic` orders the first
    // read of every ring register behind the wait.
    uint4_t tb[NT][TR][2];
    uint32_t magic = 0x64006400u;
    int ahead = 0;
    RowsCursor ic, cc;
    ic.lin = 0;
    rows_seek<TR, false>(ic, descs, nlin, b, nwg, sync, lane);
    cc.lin = 0;
    if (wave == 0) rows_seek<TR, true>(cc, descs, nlin, b, nwg, sync, lane);
    else rows_seek<TR, false>(cc, descs, nlin, b, nwg, sync, lane);

    // the buffer of this wavefront's rows in the pass the cursor is in: it ends behind them
    auto tile_rsrc = [&](const RowsCursor& c) {
      const int nt = c.tiles_of(wave, TR);
      const int row0 = c.first_of(wave) * 16;
      const int rows = nt > 0 ? min(nt * 16, c.N - row0) : 0;
      const uint64_t a = reinterpret_cast<uint64_t>(c.W + (int64_t)(nt > 0 ? row0 : 0) * c.row_w);
      return uint4_t{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, (uint32_t)(rows * c.row_w), (uint32_t)kBufferFlags};
    };

    uint4_t i_rsrc = uint4_t{0, 0, 0, (uint32_t)kBufferFlags};
    uint32_t i_voff = 0;
    auto issue = [&](uint4_t (&buf)[TR][2]) {
      if (ic.lin >= nlin) return;
      if (ic.q == 0) {
        i_rsrc = tile_rsrc(ic);
        // lane (i, kq): row i mod 8 of the half tile, scale group 4 (i / 8) + kq of the pair
        i_voff = __umul24((uint32_t)(i & 7), (uint32_t)ic.row_w) + (uint32_t)(((i >> 3) * 4 + kq) * 16);
      }
      const int rw8 = ic.row_w * 8;
      int soff = ic.q * (kRPairGroups * 16);
#pragma unroll
      for (int t = 0; t < TR; ++t) {
        // (a half tile without rows: no scalar offset against a buffer that ends before it, see direct_load16_if.  Its loads read
        // the wavefront's first rows once more, or, where it has none, zeros.)
        const int lo = soff & wq_live(soff, (int)i_rsrc.z), hi = (soff + rw8) & wq_live(soff + rw8, (int)i_rsrc.z);
        asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen nt" : "=&v"(buf[t][0]) : "v"(i_voff), "s"(i_rsrc), "s"(lo));
        asm volatile("buffer_load_dwordx4 %0, %1, %2, %3 offen nt" : "=&v"(buf[t][1]) : "v"(i_voff), "s"(i_rsrc), "s"(hi));
        soff += 2 * rw8;
      }
      ++ahead;
      rows_advance<TR, false>(ic, 1, descs, nlin, b, nwg, sync, lane);
    };

    const half2_t k1031 = {(half_t)-1031.0f, (half_t)-1031.0f};
    const half2_t k71 = {(half_t)-71.0f, (half_t)-71.0f}, sixteenth = {(half_t)0.0625f, (half_t)0.0625f};
    auto unpack = [&](uint32_t t, half2_t s2) { return as_u32((as_half2(t) + k1031) * s2); };  // of codes in bits 0 .. 3
    auto unpack4 = [&](uint32_t t, half2_t s2) { return as_u32(__builtin_elementwise_fma(as_half2(t), sixteenth, k71) * s2); };  // 4 .. 7: (1024 + 16 q) / 16 - 71

    float4_t acc[TR][R];
    int pk = -1, sk = -1;  // panels of activations / of scales taken (counted over the launch)
    int c_tr = 0;    // row tiles of this wavefront in the pass being multiplied
    int c_row0 = 0;

    auto epilogue = [&]() {
      const int lin = cc.lin;
      const int j16 = lane & 15, rq = lane >> 4;
      const half_t* bias = descs[lin].bias;
      const half_t* residual = descs[lin].residual;
      const int N = cc.N;
      const int yrows = (int)((desc_group_word(descs, lin) >> 16) & 0xffu);
      const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(descs[lin].y, 0, yrows * N * 2, kBufferFlags);
      const bool wide = (N & 3) == 0 && (((uintptr_t)descs[lin].y | (uintptr_t)bias | (uintptr_t)residual) & 7) == 0;
#pragma unroll
      for (int t = 0; t < TR; ++t) {
        if (t >= c_tr) break;
        // lane (j, rq) holds rows n0 .. n0 + 3 of activation rows j, j + 16
        const int n0 = c_row0 + 16 * t + 4 * rq;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int j = j16 + 16 * r;
          if (j < yrows && wide) {
            if (n0 < N) {
              float4_t v = acc[t][r];
              if (bias) {
                const half4_t bv = *reinterpret_cast<const half4_t*>(bias + n0);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += (float)bv[e];
              }
              half4_t h = {(half_t)v[0], (half_t)v[1], (half_t)v[2], (half_t)v[3]};
              if (residual) h = h + *reinterpret_cast<const half4_t*>(residual + (int64_t)j * N + n0);
              // device-scope store: written through, so that a counter update after it publishes it
              __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2_t, h), yr, (j * N + n0) * 2, 0, kDeviceScope);
            }
          } else if (j < yrows) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int n = n0 + e;
              if (n < N) {
                float v = acc[t][r][e];
                if (bias) v += (float)bias[n];
                half_t h = (half_t)v;
                if (residual) h = h + residual[(int64_t)j * N + n];
                __builtin_amdgcn_raw_buffer_store_b16(as_u16(h), yr, (j * N + n) * 2, 0, kDeviceScope);
              }
            }
          }
        }
      }
    };

    auto consume = [&](uint4_t (&buf)[TR][2]) {
      if (cc.q == 0) {
        c_tr = cc.tiles_of(wave, TR);
        c_row0 = cc.first_of(wave) * 16;
#pragma unroll
        for (int t = 0; t < TR; ++t)
#pragma unroll
          for (int r = 0; r < R; ++r) acc[t][r] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
      }
      if ((cc.q & 1) == 0) {
        ++pk;
        wait.until(&flags->x_ready[pk % nxb], pk + 1, 1);
      }
      if ((cc.q & 3) == 0) {
        ++sk;
        wait.until(&flags->s_ready[sk & 1], sk + 1, 2);
      }
      if (ahead == NT) asm volatile("s_waitcnt vmcnt(%1)" : "+v"(magic) : "n"((NT - 1) * LPI));
      else asm volatile("s_waitcnt vmcnt(0)" : "+v"(magic));
      // Both loads of every row tile have landed.  The chunks of the pair, put where the MFMA wants them: lanes 8 .. 15
      // of every 16 take their half of chunk 0 from the second load 8 lanes below (row_ror:8 turns a row of 16 lanes
      // by 8), lanes 0 .. 7 their half of chunk 1 from the first load 8 lanes above.  The statements depend on the wait
      // through `magic`; they are volatile so that they stay in front of the loads that refill the slot.
      uint32_t cw[TR][2][4];
#pragma unroll
      for (int t = 0; t < TR; ++t)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const uint32_t lo_in = d == 0 ? buf[t][0].x : d == 1 ? buf[t][0].y : d == 2 ? buf[t][0].z : buf[t][0].w;
          const uint32_t hi_in = d == 0 ? buf[t][1].x : d == 1 ? buf[t][1].y : d == 2 ? buf[t][1].z : buf[t][1].w;
          asm volatile("v_mov_b32_dpp %0, %2 quad_perm:[0,1,2,3] row_mask:0xf bank_mask:0xf\n\t"
                       "v_mov_b32_dpp %1, %3 quad_perm:[0,1,2,3] row_mask:0xf bank_mask:0xf\n\t"
                       "v_mov_b32_dpp %0, %3 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
                       "v_mov_b32_dpp %1, %2 row_ror:8 row_mask:0xf bank_mask:0x3 ; %4"
                       : "=&v"(cw[t][0][d]), "=&v"(cw[t][1][d])
                       : "v"(lo_in), "v"(hi_in), "v"(magic));
        }
      // the slot is free: the pair after the next one goes into it, so that two pairs are in flight while this one
      // is multiplied
      --ahead;
      issue(buf);
      if (c_tr > 0) {
        const char* const xs = xbuf + (pk % nxb) * xbuf_bytes + (kq * M + min(i, M - 1)) * 16;
        const int xr1 = (min(i + 16, M - 1) - min(i, M - 1)) * 16;  // second set of 16 activation rows
        const char* const ss = sbuf + (sk & 1) * SBUF + (wave * TROWS + i) * kRSRow + ((cc.q & 3) * kRPairGroups + kq) * 2;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          half2_t s16[TR];
#pragma unroll
          for (int t = 0; t < TR; ++t) {
            const half_t sh = *reinterpret_cast<const half_t*>(ss + t * 16 * kRSRow + u * 8);
            s16[t] = half2_t{sh, sh};
          }
          const int step = (cc.q & 1) * 2 + u;  // 128 k each within the panel
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            half8_t xb[R];
#pragma unroll
            for (int r = 0; r < R; ++r)
              xb[r] = *reinterpret_cast<const half8_t*>(xs + ((step * 4 + d) * 4 * M) * 16 + r * xr1);
#pragma unroll
            for (int t = 0; t < TR; ++t) {
              const uint32_t word = cw[t][u][d];  // (row tiles past the wavefront's share of a short pass: never stored)
              const uint32_t w8 = word >> 8;
              const uint32_t a0 = unpack(and_or(word, 0x000F000Fu, magic), s16[t]);   // (q0, q4)
              const uint32_t a1 = unpack4(and_or(word, 0x00F000F0u, magic), s16[t]);  // (q1, q5)
              const uint32_t a2 = unpack(and_or(w8, 0x000F000Fu, magic), s16[t]);     // (q2, q6)
              const uint32_t a3 = unpack4(and_or(w8, 0x00F000F0u, magic), s16[t]);    // (q3, q7)
              const half8_t aop = __builtin_bit_cast(half8_t, uint4_t{a0, a1, a2, a3});
#pragma unroll
              for (int r = 0; r < R; ++r) acc[t][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(aop, xb[r], acc[t][r], 0, 0, 0);
            }
          }
        }
      }
      const bool last = cc.q == cc.Q - 1;
      if ((cc.q & 1) == 1 || last) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wavefront's reads of the panel have returned
        if (lane == 0) __hip_atomic_fetch_add(&flags->x_taken[pk % nxb], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (((cc.q & 3) == 3 || last) && lane == 0)
          __hip_atomic_fetch_add(&flags->s_taken[sk & 1], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      if (last) {
        if (c_tr > 0) epilogue();
        if (cc.left <= kRW * TR && (descs[cc.lin].g_dep & kSignal)) {
          // the linear is complete once the stores of all 8 compute wavefronts are written through
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          int old = 0;
          int* const cnt = &flags->lin_done[cc.lin & 7];
          if (lane == 0) old = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          if (__builtin_amdgcn_readfirstlane(old) == kRW - 1 && lane == 0) {
            __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_fetch_add(sync + sync_counter_index(cc.lin, b & (kCountersPerLinear - 1)), 1, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
          }
        }
      }
      if (wave == 0) rows_advance<TR, true>(cc, 1, descs, nlin, b, nwg, sync, lane);
      else rows_advance<TR, false>(cc, 1, descs, nlin, b, nwg, sync, lane);
    };

#pragma unroll
    for (int t = 0; t < NT; ++t) issue(tb[t]);
    while (cc.lin < nlin) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (cc.lin < nlin) consume(tb[t]);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing of the ring (or of the signals) is in flight any more
    if (!use_sync) return;
    // the last compute wavefront of the last workgroup to get here clears the counters for the next launch
    int old = 0;
    if (lane == 0) old = __hip_atomic_fetch_add(&flags->exited, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (__builtin_amdgcn_readfirstlane(old) != kRW - 1) return;
    int lastwg = 0;
    if (lane == 0)
      lastwg = __hip_atomic_fetch_add(sync + sync_finished_index(nlin), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nwg - 1;
    if (__builtin_amdgcn_readfirstlane(lastwg)) {
      for (int k = lane; k < nlin * kCountersPerLinear; k += 64)
        __hip_atomic_store(sync + k * kCounterStride, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (lane == 0)
        __hip_atomic_store(sync + sync_finished_index(nlin), 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return;
  }

  if (wave < kRW + kRXW) {
    // ====================== x wavefronts: a panel of activations -> LDS ======================
    const int xw = wave - kRW;
    bool aborted = false;
    auto wait_for = [&](int dep) {
      if (aborted) return;
      const long long t0 = wall_clock64();
      while (true) {
        int v = 0;
        if (lane < kCountersPerLinear)
          v = __hip_atomic_fetch_add(sync + sync_counter_index(dep, lane), 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        v += __shfl_xor(v, 1, 64);
        v += __shfl_xor(v, 2, 64);
        v += __shfl_xor(v, 4, 64);
        if (__builtin_amdgcn_readfirstlane(v) >= group_size(desc_group_word(descs, dep), nwg)) break;  // every member of its group
        if (wall_clock64() - t0 > spin_limit) {
          aborted = true;
          if (lane == 0)
            __hip_atomic_store(sync + sync_error_index(nlin), dep + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
        __builtin_amdgcn_s_sleep(4);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    };
    constexpr int PPR = kRPG * 4;  // 16-byte pieces (8 activations) per row and panel
    constexpr int UX = 32;         // loads in flight per lane: a whole panel of 32 rows
    RowsCursor xc;
    xc.lin = 0;
    rows_seek<TR, false>(xc, descs, nlin, b, nwg, sync, lane);
    int pk = 0;
    int confirmed = -1;
    while (xc.lin < nlin) {
      if (pk % kRXW == xw) {
        const int xslot = pk % nxb;
        if (pk >= nxb) wait.until(&flags->x_taken[xslot], kRW * (pk / nxb), 4);
        const int j = xc.lin;
        const int dep = (int)((descs[j].g_dep >> 16) & 0x7fffu) - 1;
        if (dep >= 0 && dep != confirmed) {
          wait_for(dep);
          confirmed = dep;
        }
        const int K8 = xc.G << 2;
        const int xrows = (int)((desc_group_word(descs, j) >> 16) & 0xffu);
        const __amdgpu_buffer_rsrc_t xr =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(descs[j].x), 0, xrows * K8 * 16, kBufferFlags);
        char* const xdst = xbuf + xslot * xbuf_bytes;
        const int p0 = xc.q * (kRPairGroups * 4);  // the panel's first piece within a row
        const int total = M * PPR;
        for (int base = 0; base < total; base += 64 * UX) {
          uint4_t v[UX];
#pragma unroll
          for (int t = 0; t < UX; ++t) {
            const int idx = base + t * 64 + lane;
            const int row = idx / PPR, o = idx & (PPR - 1);
            const int go = p0 + o;
            v[t] = uint4_t{0, 0, 0, 0};
            const int src = min(row, xrows - 1);
            if (idx < total && go < K8)
              v[t] = dep >= 0 ? __builtin_amdgcn_raw_buffer_load_b128(xr, (src * K8 + go) * 16, 0, kDeviceScope)
                              : __builtin_amdgcn_raw_buffer_load_b128(xr, (src * K8 + go) * 16, 0, 0);
          }
#pragma unroll
          for (int t = 0; t < UX; ++t) {
            const int idx = base + t * 64 + lane;
            if (idx < total) {
              const int row = idx / PPR, o = idx & (PPR - 1);
              const uint32_t in[4] = {v[t].x, v[t].y, v[t].z, v[t].w};
              uint32_t p[4];
              pair_i_i4(in, p);  // p[e] = (x_e, x_{e+4})
              // piece o: scale group g = o / 4 of the panel, dword d = o % 4 of it; step g / 4, lane quarter g % 4
              const int g = o >> 2, d = o & 3;
              char* dst = xdst + ((((g >> 2) * 4 + d) * 4 + (g & 3)) * M + row) * 16;
              *reinterpret_cast<uint4_t*>(dst) = uint4_t{p[0], p[1], p[2], p[3]};
            }
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (lane == 0) __hip_atomic_store(&flags->x_ready[xslot], pk + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      ++pk;
      rows_advance<TR, false>(xc, kRPG / kRPairGroups, descs, nlin, b, nwg, sync, lane);
    }
    return;
  }

  // ====================== scale wavefront: the scales of a pass, 1024 k at a time -> LDS ======================
  {
    constexpr int PPR = kRSPG / 8;              // 16-byte pieces (8 scales) per row and panel
    constexpr int LP = kRW * TROWS * PPR / 64;  // pieces per lane and panel
    RowsCursor sc;
    sc.lin = 0;
    rows_seek<TR, false>(sc, descs, nlin, b, nwg, sync, lane);
    int sk = 0;
    while (sc.lin < nlin) {
      const int sslot = sk & 1;
      const int g0 = sc.q * kRPairGroups;  // first scale group of the panel
      const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<char*>(sc.S), 0, (int)min((int64_t)sc.N * sc.G * 2, (int64_t)0x7fffffff), kBufferFlags);
      uint4_t v[LP];
#pragma unroll
      for (int t = 0; t < LP; ++t) {
        const int idx = t * 64 + lane;
        const int rr = idx / PPR, pc = idx % PPR;
        const int w = rr / TROWS, r = rr % TROWS;
        const int row = sc.first_of(w) * 16 + r;
        v[t] = uint4_t{0, 0, 0, 0};  // rows past the wavefront's or past N, groups past K: a zero scale
        if (r < sc.tiles_of(w, TR) * 16 && row < sc.N && g0 + pc * 8 < sc.G)
          v[t] = __builtin_amdgcn_raw_buffer_load_b128(sr, (row * sc.G + g0 + pc * 8) * 2, 0, 0);
      }
      // the buffer is free once every compute wavefront has left the panel that used it before
      if (sk >= 2) wait.until(&flags->s_taken[sslot], kRW * (sk / 2), 5);
#pragma unroll
      for (int t = 0; t < LP; ++t) {
        const int idx = t * 64 + lane;
        const int rr = idx / PPR, pc = idx % PPR;
        *reinterpret_cast<uint4_t*>(sbuf + sslot * SBUF + rr * kRSRow + pc * 16) = v[t];
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      ++sk;
      if (lane == 0) __hip_atomic_store(&flags->s_ready[sslot], sk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      rows_advance<TR, false>(sc, kRSPG / kRPairGroups, descs, nlin, b, nwg, sync, lane);
    }
  }
}

// ------------------------------------------------------------------ host side
// the kernel a list of M activation rows runs: chunks per wavefront and tile, tile rows / 16
struct BatchShape {
  bool wide;
  int SP, RT;
};
// The shapes there are.  An item of a panel of 2048 k suits K up to there, since a panel is walked whole, and that of 4096 k
// spends least on hand-overs; two row tiles per item halve the hand-overs where there are enough rows.  (Panels of 2048 k
// with the operands of up to 8 rows: within 2 % of those of up to 16 at M = 2 and 8, so they are not there.)
static const BatchShape kBatchShapes[] = {{false, 2, 2}, {false, 2, 1}, {true, 1, 2}, {true, 1, 1}};
constexpr int kBatchShapeCount = sizeof(kBatchShapes) / sizeof(kBatchShapes[0]);

constexpr size_t kBatchLds = 160 * 1024;
static size_t batch_lds_bytes(BatchShape s, int M, int nxb, int ring, int acc_tiles) {
  return sizeof(BatchFlags) + (size_t)nxb * M * batch_panel_groups(s.SP) * 64 + (size_t)ring * batch_scale_slot_bytes(s.SP, s.RT) +
         (size_t)ring * batch_partial_slot_bytes(s.wide, s.RT) + (size_t)acc_tiles * batch_kept_bytes(s.RT);
}

// Which group of workgroups runs which linear.  Every workgroup needs all M x K activations of a linear
// it takes part in: with 256 workgroups on a 4096-row linear that is twice the weights at M = 8.  So a list is run by 2^g
// groups side by side, each linear by one group (group = workgroup index mod 2^g, which is one XCD for
// g = 3: the activations then stay in that XCD's L2): a workgroup sees 1 / 2^g of the linears and 2^g times
// as many rows of each.  Linears go, in list order, to the group that can start them first (a consumer
// not before its producer has ended), with the duration of a linear estimated (batch_linear_cost); g is the best of
// 0 .. 4 by that estimate, and so is the shape.
struct BatchGroupPlan {
  std::vector<int> group;
  double makespan = 0.0;
};

// chunks a workgroup with `tiles` tiles of a linear walks them in (each chunk loads every panel of activations again)
static int batch_chunks(int tiles, int panels, int chunk) { return panels > 1 && tiles > chunk ? (tiles + chunk - 1) / chunk : 1; }

// How long a workgroup of a group of `ncu` takes for linear i, in units near a microsecond: an item, a panel of activations
// (beside which the items run, but little of it is hidden where LDS holds one panel only), a linear, and the wait for a
// producer.  Fitted to the launches of 40 lists (M = 2 .. 16, hidden 1024 .. 8192, 1 .. 32 layers) under every shape and
// number of groups, 912 in all: the plan that the estimate picks is 1.0 % slower than the fastest one on average, 9 % at
// most (M = 8, hidden 8192, ffn 28672, three layers).  Against bytes alone, by which a list was planned before: hidden 2048, ffn
// 5632, 32 layers, M = 8 381 -> 218 us, one layer 34.4 -> 20.6; over 45 lists, M = 2 .. 16, 21 % with the products above.
// (64 KiB items of a linear of several panels take longer: all workgroups read the same half of its rows' bytes.)
constexpr double kBatchAfterProducer = 22.0;
static double batch_linear_cost(const wq_gemv_list* l, int i, int ncu, BatchShape s, int fit) {
  const GemvListDesc& g = l->descs[i];
  const int G = (int)(g.g_dep & 0xffffu);
  const int trows = 16 * s.RT;
  const int tiles = (int)((((int64_t)g.N + trows - 1) / trows + ncu - 1) / ncu);  // of one workgroup
  const int panels = (G + batch_panel_groups(s.SP) - 1) / batch_panel_groups(s.SP);
  const int chunks = batch_chunks(tiles, panels, fit), kept = panels > 1 ? std::min(tiles, fit) : 0;
  const double item = (0.41 + 0.44 * s.RT * s.SP) * (s.RT * s.SP == 4 && panels > 1 ? 1.2 : 1.0), x = 1.15 + 0.34 * l->M * s.SP;
  const double seen = batch_lds_bytes(s, l->M, 2, 2, kept) <= kBatchLds ? 0.1 : 0.45;
  return 4.1 + chunks * panels * std::max(x, (double)tiles / chunks * item + seen * x);
}

// A SHORT list has too few linears for equal groups to be both many (so that few workgroups load a linear's
// activations) and busy.  Its linears share the 8 XCDs instead, level by level: the linears of a dependency
// level (level = 1 + the level of the producer) run side by side, each on a set of XCDs in proportion to what
// it costs, every set at least one XCD.  cost(i, workgroups of the group) as above.
struct MaskPlan {
  bool ok = false;
  std::vector<uint8_t> mask;  // XCDs of linear i
  double makespan = 0.0;
};
template <class Cost>
static MaskPlan plan_xcd_masks(const wq_gemv_list* l, Cost cost, double after_producer = 0.0) {
  MaskPlan plan;
  if (l->blocks % 8 != 0 || l->n > 64) return plan;
  const int per_xcd = l->blocks / 8;
  std::vector<int> level(l->n, 0);
  int levels = 0;
  for (int i = 0; i < l->n; ++i) {
    const int dep = (int)((l->descs[i].g_dep >> 16) & 0x7fffu) - 1;
    level[i] = dep >= 0 ? level[dep] + 1 : 0;
    levels = std::max(levels, level[i] + 1);
  }
  plan.mask.assign(l->n, 0);
  for (int lv = 0; lv < levels; ++lv) {
    std::vector<int> who;
    for (int i = 0; i < l->n; ++i)
      if (level[i] == lv) who.push_back(i);
    if (who.size() > 8) return plan;  // a long list: equal groups
    std::vector<int> k(who.size(), 1);
    for (int left = 8 - (int)who.size(); left > 0; --left) {  // one more XCD to whoever takes longest
      size_t worst = 0;
      for (size_t a = 1; a < who.size(); ++a)
        if (cost(who[a], per_xcd * k[a]) > cost(who[worst], per_xcd * k[worst])) worst = a;
      ++k[worst];
    }
    int next = 0;
    for (size_t a = 0; a < who.size(); ++a) {
      plan.mask[who[a]] = (uint8_t)(((1u << k[a]) - 1u) << next);
      next += k[a];
    }
  }
  // How long that takes: an XCD walks its linears in list order, whatever their level, so one that waits for a producer holds
  // up what follows it (as levels one behind the other the estimate chose sets that took up to 1.4 times as long as groups).
  double free_at[8] = {};
  std::vector<double> end(l->n, 0.0);
  for (int i = 0; i < l->n; ++i) {
    const int dep = (int)((l->descs[i].g_dep >> 16) & 0x7fffu) - 1;
    const double ready = dep >= 0 ? end[dep] + after_producer : 0.0, dur = cost(i, per_xcd * __builtin_popcount(plan.mask[i]));
    for (int x = 0; x < 8; ++x) {
      if (!((plan.mask[i] >> x) & 1)) continue;
      free_at[x] = std::max(free_at[x], ready) + dur;
      end[i] = std::max(end[i], free_at[x]);
    }
    plan.makespan = std::max(plan.makespan, end[i]);
  }
  plan.ok = true;
  return plan;
}

static BatchGroupPlan batch_assign_groups(const wq_gemv_list* l, int gl, BatchShape s, int fit) {
  const int groups = 1 << gl, ncu = l->blocks >> gl;
  BatchGroupPlan plan;
  plan.group.resize(l->n);
  std::vector<double> free_at(groups, 0.0), end(l->n, 0.0);
  for (int i = 0; i < l->n; ++i) {
    const GemvListDesc& g = l->descs[i];
    const double dur = batch_linear_cost(l, i, ncu, s, fit);
    const int dep = (int)((g.g_dep >> 16) & 0x7fffu) - 1;
    const double ready = dep >= 0 ? end[dep] + kBatchAfterProducer : 0.0;
    int best = 0;
    for (int c = 1; c < groups; ++c) {
      const double sb = std::max(free_at[best], ready), sc = std::max(free_at[c], ready);
      if (sc < sb || (sc == sb && free_at[c] > free_at[best])) best = c;  // earliest start, then least idle time
    }
    plan.group[i] = best;
    end[i] = std::max(free_at[best], ready) + dur;
    free_at[best] = end[i];
  }
  for (double f : free_at) plan.makespan = std::max(plan.makespan, f);
  return plan;
}

// the kernel that walks the tiles of a linear in chunks carries more loop state: only where a list needs it
typedef void (*batch_kernel_t)(const GemvListDesc*, int, int*, long long, int, int, int, int, int);
static batch_kernel_t batch_kernel(int shape, bool chunked) {
  switch (shape) {
    case 0: return chunked ? q4g32_batch_list_kernel<false, 2, 2, true> : q4g32_batch_list_kernel<false, 2, 2, false>;
    case 1: return chunked ? q4g32_batch_list_kernel<false, 2, 1, true> : q4g32_batch_list_kernel<false, 2, 1, false>;
    case 2: return chunked ? q4g32_batch_list_kernel<true, 1, 2, true> : q4g32_batch_list_kernel<true, 1, 2, false>;
    default: return chunked ? q4g32_batch_list_kernel<true, 1, 1, true> : q4g32_batch_list_kernel<true, 1, 1, false>;
  }
}

// ---- lists of more than 16 activation rows: q4g32_batch_rows_kernel
constexpr int kRowsTR = 4;  // row tiles of a wave tile: 64 rows
static size_t rows_lds_bytes(int M, int nxb) {
  return sizeof(RowsFlags) + (size_t)nxb * M * kRPG * 64 + 2 * (size_t)kRW * 16 * kRowsTR * kRSRow;
}

// as batch_assign_groups, with the duration of a linear from the passes a workgroup makes over its wave tiles
// (every pass loads all activations; a pass of fewer than 8 wave tiles takes as long as a full one)
// pass by pass: all activations, and the time of 8 wavefronts x TR row tiles however few rows the pass holds (a
// wavefront unpacks and multiplies TR row tiles per pair either way; measured on the 32-layer Llama-2-7B stack,
// M = 32: 16 groups, where the 4096-row linears make one pass of 32 rows per wavefront, 1.19 ms; 32 groups 0.945 ms)
static double rows_linear_cost(const wq_gemv_list* l, int i, int ncu) {
  const GemvListDesc& g = l->descs[i];
  const double K = (double)(g.g_dep & 0xffffu) * 32.0;
  const int64_t tiles = ((int64_t)g.N + 15) / 16;   // row tiles
  const int64_t left = (tiles + ncu - 1) / ncu;      // of the workgroup with most
  const double passes = (double)((left + kRW * kRowsTR - 1) / (kRW * kRowsTR));
  return 4096.0 + passes * (kRW * kRowsTR * 16.0 * K * (0.5 + 1.0 / 16.0) + l->M * K * 2.0);
}

static BatchGroupPlan rows_assign_groups(const wq_gemv_list* l, int gl) {
  const int groups = 1 << gl, ncu = l->blocks >> gl;
  BatchGroupPlan plan;
  plan.group.resize(l->n);
  std::vector<double> free_at(groups, 0.0), end(l->n, 0.0);
  for (int i = 0; i < l->n; ++i) {
    const GemvListDesc& g = l->descs[i];
    const double dur = rows_linear_cost(l, i, ncu);
    const int dep = (int)((g.g_dep >> 16) & 0x7fffu) - 1;
    const double ready = dep >= 0 ? end[dep] : 0.0;
    int best = 0;
    for (int c = 1; c < groups; ++c) {
      const double sb = std::max(free_at[best], ready), sc = std::max(free_at[c], ready);
      if (sc < sb || (sc == sb && free_at[c] > free_at[best])) best = c;
    }
    plan.group[i] = best;
    end[i] = std::max(free_at[best], ready) + dur;
    free_at[best] = end[i];
  }
  for (double f : free_at) plan.makespan = std::max(plan.makespan, f);
  return plan;
}

static int rows_list_plan(wq_gemv_list* l) {
  for (int i = 0; i < l->n; ++i)  // the scales are addressed with 32-bit offsets
    if ((int64_t)l->descs[i].N * (l->descs[i].g_dep & 0xffffu) * 2 >= (1ll << 31))
      return fail(WQ_EUNSUPPORTED, "wq_q4g32_gemv_list_create: linear %d: with more than 16 rows of activations the scales must stay below 2 GiB", i);
  l->batch_rows = true;
  l->threads = kRThreads;
  l->blocks = std::min(cu_count(), 32768);
  const size_t budget = 160 * 1024;
  int nxb = kRMaxXBuf;
  while (nxb > 1 && rows_lds_bytes(l->M, nxb) > budget) --nxb;
  if (rows_lds_bytes(l->M, nxb) > budget)
    return fail(WQ_EUNSUPPORTED, "wq_q4g32_gemv_list_create: %d rows of activations do not fit the LDS", l->M);
  int best_gl = -1;
  BatchGroupPlan best;
  for (int gl = 0; gl <= 6; ++gl) {
    if (l->blocks % (1 << gl) != 0 || (l->blocks >> gl) < 1) break;
    BatchGroupPlan p = rows_assign_groups(l, gl);
    if (best_gl < 0 || p.makespan < best.makespan * 0.98) {
      best_gl = gl;
      best = std::move(p);
    }
  }
  int groups = 1 << best_gl;
  const MaskPlan mp = plan_xcd_masks(l, [&](int i, int ncu) { return rows_linear_cost(l, i, ncu); });
  if (mp.ok && mp.makespan < best.makespan * 0.98) {
    for (int i = 0; i < l->n; ++i) {
      GemvListDesc& g = l->descs[i];
      const int ncu = (l->blocks / 8) * __builtin_popcount(mp.mask[i]);
      const int64_t tiles = ((int64_t)g.N + 15) / 16;  // row tiles
      g.q = (int32_t)(tiles / ncu);
      g.rem = (uint16_t)(tiles % ncu);
      g.off = 0;
      g.gmod_log2 = 0x80;
      g.gidx = mp.mask[i];
    }
    groups = 0;  // (sets of XCDs)
  } else {
    const int ncu = l->blocks >> best_gl;
    std::vector<int64_t> off(groups, 0);
    for (int i = 0; i < l->n; ++i) {
      GemvListDesc& g = l->descs[i];
      const int c = best.group[i];
      const int64_t tiles = ((int64_t)g.N + 15) / 16;  // row tiles
      g.q = (int32_t)(tiles / ncu);
      g.rem = (uint16_t)(tiles % ncu);
      g.off = (uint16_t)off[c];
      off[c] = (off[c] + tiles) % ncu;
      g.gmod_log2 = (uint8_t)best_gl;
      g.gidx = (uint8_t)c;
    }
  }
  l->batch_groups = groups;
  l->batch_nxb = nxb;
  l->batch_ring = 2;
  l->batch_acc_tiles = 0;
  l->batch_chunked = false;
  l->lds = rows_lds_bytes(l->M, nxb);
  const void* kern = reinterpret_cast<const void*>(q4g32_batch_rows_kernel<kRowsTR, 2>);
  static DynamicLdsLimit limit;
  if (limit.ensure(kern, (int)l->lds) != hipSuccess)
    return fail(WQ_EDEVICE, "wq_q4g32_gemv_list_create: hipFuncSetAttribute failed");
  int resident = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&resident, kern, l->threads, l->lds) != hipSuccess || resident < 1)
    return fail(WQ_EDEVICE, "wq_q4g32_gemv_list_create: the workgroup does not fit a CU (%zu bytes of LDS)", l->lds);
  return WQ_OK;
}

// a list as one of the shapes would run it
struct BatchPlan {
  double makespan = -1.0;  // < 0: not possible
  int gl = 0;              // 2^gl groups, or (masks) sets of XCDs
  bool masks = false, chunked = false;
  int acc_tiles = 0;
  std::vector<int> group;
  std::vector<uint8_t> mask;
};
static BatchPlan batch_plan(const wq_gemv_list* l, BatchShape s) {
  const int trows = 16 * s.RT;
  BatchPlan best;
  // the sums kept between panels must fit beside one panel of activations and a ring of 2: else the tiles of
  // a linear are walked in chunks of what fits, at the price of loading the activations once per chunk
  const size_t base = batch_lds_bytes(s, l->M, 1, 2, 0);
  if (base + 4 * batch_kept_bytes(s.RT) > kBatchLds) return best;
  const int fit = (int)((kBatchLds - base) / (size_t)batch_kept_bytes(s.RT));
  auto kept = [&](int i, int ncu) {  // tiles whose sums a workgroup keeps for linear i
    const int64_t tiles = ((int64_t)l->descs[i].N + trows - 1) / trows;
    return (int)(l->descs[i].g_dep & 0xffffu) > batch_panel_groups(s.SP) ? (int)((tiles + ncu - 1) / ncu) : 0;
  };
  for (int gl = 0; gl <= 4; ++gl) {
    if (l->blocks % (1 << gl) != 0 || (l->blocks >> gl) < 1) break;
    int acc_tiles = 0;
    for (int i = 0; i < l->n; ++i) acc_tiles = std::max(acc_tiles, kept(i, l->blocks >> gl));
    const int chunk = std::min(acc_tiles, fit);
    BatchGroupPlan p = batch_assign_groups(l, gl, s, fit);
    if (best.makespan < 0 || p.makespan < best.makespan * 0.98) {
      best.makespan = p.makespan;
      best.gl = gl;
      best.group = std::move(p.group);
      best.acc_tiles = chunk;
      best.chunked = chunk < acc_tiles;
    }
  }
  // a short list: sets of XCDs in proportion to the linears' cost (plan_xcd_masks), if the estimate says so
  MaskPlan mp = plan_xcd_masks(l, [&](int i, int ncu) { return batch_linear_cost(l, i, ncu, s, fit); }, kBatchAfterProducer);
  if (mp.ok && (best.makespan < 0 || mp.makespan <= best.makespan * 1.0005)) {  // (at a tie the sets)
    int acc_tiles = 0;
    for (int i = 0; i < l->n; ++i) acc_tiles = std::max(acc_tiles, kept(i, (l->blocks / 8) * __builtin_popcount(mp.mask[i])));
    best.makespan = mp.makespan;
    best.masks = true;
    best.mask = std::move(mp.mask);
    best.acc_tiles = std::min(acc_tiles, fit);
    best.chunked = best.acc_tiles < acc_tiles;
  }
  return best;
}

int batch_list_plan(wq_gemv_list* l) {
  if (l->M > 16) return rows_list_plan(l);
  l->threads = kBThreads;
  l->blocks = std::min(cu_count(), 32768);
  BatchPlan best;
  for (int i = 0; i < kBatchShapeCount; ++i) {
    if (!kBatchShapes[i].wide && l->M > 8) continue;
    BatchPlan p = batch_plan(l, kBatchShapes[i]);
    if (p.makespan >= 0 && (best.makespan < 0 || p.makespan < best.makespan)) {
      best = std::move(p);
      l->batch_shape = i;
    }
  }
  if (best.makespan < 0)
    return fail(WQ_EUNSUPPORTED, "wq_q4g32_gemv_list_create: %d rows of activations do not fit the LDS", l->M);
  const BatchShape s = kBatchShapes[l->batch_shape];
  const int groups = 1 << best.gl;
  std::vector<int64_t> off(groups, 0);
  for (int i = 0; i < l->n; ++i) {
    GemvListDesc& g = l->descs[i];
    const int ncu = best.masks ? (l->blocks / 8) * __builtin_popcount(best.mask[i]) : l->blocks >> best.gl;
    const int64_t tiles = ((int64_t)g.N + 16 * s.RT - 1) / (16 * s.RT);
    g.q = (int32_t)(tiles / ncu);
    g.rem = (uint16_t)(tiles % ncu);
    g.off = 0;
    g.gmod_log2 = best.masks ? 0x80 : (uint8_t)best.gl;
    g.gidx = best.masks ? best.mask[i] : (uint8_t)best.group[i];
    if (!best.masks) {
      int64_t& o = off[best.group[i]];
      g.off = (uint16_t)o;
      o = (o + tiles) % ncu;
    }
  }
  l->batch_groups = best.masks ? 0 : groups;
  l->batch_acc_tiles = best.acc_tiles;
  l->batch_chunked = best.chunked;
  // two panels of activations in LDS if they fit, then a ring of 4 items
  for (int c : {0, 1, 2, 3}) {
    l->batch_nxb = c < 2 ? 2 : 1;
    l->batch_ring = c % 2 ? 2 : 4;
    l->lds = batch_lds_bytes(s, l->M, l->batch_nxb, l->batch_ring, best.acc_tiles);
    if (l->lds <= kBatchLds) break;
  }
  const void* kern = reinterpret_cast<const void*>(batch_kernel(l->batch_shape, best.chunked));
  // several lists share a kernel: the limit only ever grows
  static DynamicLdsLimit limits[kBatchShapeCount][2];
  if (limits[l->batch_shape][best.chunked ? 1 : 0].ensure(kern, (int)l->lds) != hipSuccess)
    return fail(WQ_EDEVICE, "wq_q4g32_gemv_list_create: hipFuncSetAttribute failed");
  int resident = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&resident, kern, l->threads, l->lds) != hipSuccess || resident < 1)
    return fail(WQ_EDEVICE, "wq_q4g32_gemv_list_create: the workgroup does not fit a CU (%zu bytes of LDS)", l->lds);
  return WQ_OK;
}

int batch_list_launch(wq_gemv_list* l, hipStream_t stream) {
  const GemvListDesc* table = (const GemvListDesc*)l->table;
  const int use_sync = l->deps > 0 ? 1 : 0;
  if (l->batch_rows) {
    WQ_LAUNCH("wq_q4g32_gemv_list_run", (q4g32_batch_rows_kernel<kRowsTR, 2>), dim3((unsigned)l->blocks), dim3((unsigned)l->threads), l->lds,
              stream, table, l->n, l->sync, l->spin_limit, l->M, l->batch_nxb, use_sync);
    return WQ_OK;
  }
  // chunk: at least 1 (a list without a linear of several panels keeps no sums)
  WQ_LAUNCH("wq_q4g32_gemv_list_run", batch_kernel(l->batch_shape, l->batch_chunked), dim3((unsigned)l->blocks), dim3((unsigned)l->threads), l->lds,
            stream, table, l->n, l->sync, l->spin_limit, l->M, l->batch_nxb, l->batch_ring, std::max(l->batch_acc_tiles, 1),
            use_sync);
  return WQ_OK;
}

}  // namespace wq
