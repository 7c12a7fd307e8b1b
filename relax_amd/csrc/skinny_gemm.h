// Small-batch weight-streaming GEMM (2 <= M <= 64) shared by both weight formats.
//
// At small M a quantized linear layer is still a weight stream (HBM-bound), but the
// products are done by the matrix cores so that all M rows share ONE pass over the
// weights (the GEMV kernels re-read the weights every few rows and pay VALU work per
// row).  This is the counterpart of the reference's dlight LowBatchGEMV rule
// (python/tvm/dlight/gpu/low_batch_gemv.py).
//
// Work split.  A workgroup (WAVES wavefronts, arranged NW x KW) owns 16*NW output
// columns and all M rows.  Wavefront (nw, kw) owns columns n0 + 16*nw .. +15 and the
// K-steps kw, kw + KW, kw + 2*KW, ... of 128 k each.  One step of one wavefront is
// 4*TM MFMA 16x16x32: lane (j, kq) holds, for both operands, the 32 consecutive k
// 128*step + 32*kq .. +31 of column j (row j of the activations), of which MFMA t takes
// k 8t .. 8t+7.  The weight format (a Policy) says where those 32 codes live, how
// many 16-byte pieces they are and how they unpack into the four B operands, in
// natural k order, so the activations need no rearrangement.
//
// Everything travels global -> LDS with direct loads into a ring of `stages` slots,
// `stages - 1` steps ahead: per step the rows x 128 activation slab of each kw
// (shared by the NW wavefronts of that kw, each loading a part), and per wavefront
// its codes and scales (or, where the policy and K allow, all scales of the column block
// once, ahead of the ring).  A wavefront waits for its own loads with s_waitcnt vmcnt(n);
// when NW > 1 one s_barrier per step makes the shared slab visible.  The KW partial
// sums of a column block meet in LDS at the end.
//
// What bounds it: per 16 columns every workgroup re-reads all of the activations
// (from L2), and unpacking costs about two VALU operations per weight, so eight
// wavefronts per workgroup (two per SIMD) are used to overlap one wavefront's
// unpacking with another's loads, and NW grows with M and N to cut the re-reads.
#ifndef RELAX_AMD_CSRC_SKINNY_GEMM_H_
#define RELAX_AMD_CSRC_SKINNY_GEMM_H_

#include <type_traits>

#include "tuning.h"
#include "wq_device.h"
#include "wq_host.h"

namespace wq {

#define WQ_SK_WAITCNT_VM(n) __builtin_amdgcn_s_waitcnt(((n)&0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0xF << 8))

// A Policy provides
//   kPieces            16-byte pieces of codes per lane and step (32 k)
//   kScaleDma          true: a scale per lane and step, fetched as the 4-byte pair that holds it
//   Args, Lane         kernel argument block / per-lane state
//   init(lane, args, n, K, N)
//   w_addr(lane, k0, p)        address of piece p of the 32 codes starting at k0 (k0 % 32 == 0)
//   s_addr(lane, k0)           4-byte aligned address of the pair holding the scale for k0   (kScaleDma)
//   Scale                      what dequant needs besides the codes (half_t, or scale and zero point)
//   pick_scale(lane, pair, kq) the lane's Scale from that pair                               (kScaleDma)
//   const_scale(lane)          the lane's Scale                                              (!kScaleDma)
//   null_scale()               a Scale that turns every code into an exact zero (weights past K)
//   dequant(pieces, s, out[4]) -> B operands of MFMA 0..3 (k 8t .. 8t+7 each), scaled
//   s_pair_addr(lane, k0)      like s_addr, for every policy (a fixed scale: the pair that holds it)
//   kCanScaleBlock             true (needs kScaleDma): the scales of a column are 2-byte values, contiguous
//                              along K, one per 32 k; where scale_block_ok(args, K) the ring kernel may
//                              fetch all scales of a column block once, 16 bytes per lane, instead of a
//                              pair per lane and step
//                              (then scale g of the lane's column lies at s_lane(lane) + 2 g)
//   scale_block_ok(args, K)    host: every 8 scales of a column are 16 aligned bytes      (kCanScaleBlock)
//   pair_aligned(args)         host: whether those pairs are 4-byte aligned
//   kStepStride                bytes between a lane's pieces of consecutive steps (128 k)
//   s_lane(lane), s_rel(lane, k0)   s_addr(lane, k0) as a pointer and a 32-bit offset from it           (kScaleDma)
//   s_reach(args, N, K)        host: no such offset inside 16 columns goes beyond this
//   s_step(N)                  optional: bytes between a lane's scales of consecutive steps, where they lie evenly (then
//                              s_reach has room for 8 steps past K)
// and, for weights that are not rounded (up to 8 rows, kPieces == 1),
//   codes8(word)               the codes of a word of codes as halves, exact (8 consecutive k); the products of a
//                              group of 32 k are summed alone and scaled in fp32
constexpr int kScaleBlockMaxK = 11264;  // a column block's scales for all of K stay in LDS: K bytes
inline int scale_block_stride(int K) { return ((K + 1023) >> 10) << 10; }

template <class P, class = void>
struct GroupSums : std::false_type {};
template <class P>
struct GroupSums<P, std::void_t<decltype(&P::codes8)>> : std::true_type {};

// Policy::kColumnScale = true: one scale per column, which the sums take and not the weights (dequant gives the codes as they are;
// Policy::kZeroCodes is a word of codes that are zero)
// the codes past K, whose weights have to be zero
template <class P>
__device__ __forceinline__ void zero_codes(uint4_t (&pieces)[P::kPieces]) {
#pragma unroll
  for (int p = 0; p < P::kPieces; ++p) pieces[p] = uint4_t{P::kZeroCodes, P::kZeroCodes, P::kZeroCodes, P::kZeroCodes};
}

// Policy::kXreg = false: no form with the activations in registers here
template <class P, class = void>
struct UsesXreg : std::true_type {};
template <class P>
struct UsesXreg<P, std::void_t<decltype(P::kXreg)>> : std::bool_constant<P::kXreg> {};

// Policy::kOddStart = true: s_rel may be -2 (the pair begins in front of the column)
template <class P, class = void>
struct OddStart : std::false_type {};
template <class P>
struct OddStart<P, std::void_t<decltype(P::kOddStart)>> : std::bool_constant<P::kOddStart> {};

template <class P, class = void>
struct ScaleStep : std::false_type {};
template <class P>
struct ScaleStep<P, std::void_t<decltype(&P::s_step)>> : std::true_type {};

// bits 0 .. n - 1 of `groups` groups, of which those up to K exist
__device__ __forceinline__ uint32_t live_groups(int k0, int K, int groups) {
  const int n = min(max((K - k0) >> 5, 0), groups);
  return n >= 32 ? ~0u : (1u << n) - 1u;
}

// One step of 128 k with the scales outside the products (GroupSums).  MFMA g takes group g whole: a quarter kq of
// the wavefront brings k 32g + 8kq .. + 7, so lane (j, kq) reads the word kq of the piece that lane (j, g) fetched
// (4 bytes a lane, the 64 of them contiguous), and the scale that lane fetched.  a(g) is the A operand; groups past K,
// whose bit first + g of `live` is clear, get a zero scale (a mask: a branch would keep the reads from being issued
// together).
template <class Policy, class AOp>
__device__ __forceinline__ void mul_group_sums(float4_t& acc, const typename Policy::Lane& pl, const unsigned char* pieces,
                                               const unsigned char* pairs, int lj, int kq, uint32_t live, int first, AOp a) {
  static_assert(Policy::kPieces == 1 && Policy::kScaleDma);
  const uint32_t* const w = reinterpret_cast<const uint32_t*>(pieces + lj * 16 + kq * 4);
  const uint32_t* const p = reinterpret_cast<const uint32_t*>(pairs + lj * 4);
  uint32_t word[4], pair[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    word[g] = w[g * 64];
    pair[g] = p[g * 16] & (uint32_t)((int32_t)(live << (31 - first - g)) >> 31);
  }
  half8_t aop[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) aop[g] = a(g);
  float s[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) s[g] = (float)Policy::pick_scale(pl, as_half2(pair[g]), g);
  float4_t sum[4];
#pragma unroll
  for (int g = 0; g < 4; ++g)
    sum[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(aop[g], Policy::codes8(word[g]), float4_t{}, 0, 0, 0);
#pragma unroll
  for (int g = 0; g < 4; ++g) {
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = fmaf(s[g], sum[g][r], acc[r]);
  }
}

// Position of the 16-byte chunk c of row r of a slab (256 bytes a row): c ^ slab_swizzle(r).  LDS serves a 16-byte read by
// lanes 0 .. 3, 12 .. 15, 20 .. 27 and by 4 .. 11, 16 .. 19, 28 .. 31 together (and the same from 32 on), and an operand's
// lanes 0 .. 15 / 16 .. 31 take chunks 4 apart of rows 0 .. 15: rows 0 .. 3 and 12 .. 15 must not differ in the bit that
// tells those chunks apart from what rows 4 .. 11 hold.  With r itself every read met another one in its banks (q4f16_1,
// N = 12288, K = 4096, M = 19: 786 of 1757 thousand LDS cycles; now none of 971).
__device__ __forceinline__ int slab_swizzle(int r) { return (r & 3) | ((r & 8) >> 1) | ((r & 8) ^ ((r & 4) << 1)); }

// Byte offsets inside the activations and inside 16 columns of weights fit 31 bits below this K; from here on, and where
// the scales reach further, one arrangement with 64-bit addresses serves (WIDE).
constexpr int64_t kSkinnyMaxK = 1 << 23;
constexpr uint32_t kOutside = 0x80000000u;  // bytes that a descriptor spans; an offset from here on brings zeros
static __device__ const uint4_t kZeroChunk = {0, 0, 0, 0};  // ... as this does for loads without a descriptor
__device__ __forceinline__ void direct_load16(const char* base, wq_lptr_t dst, uint32_t off, int step_off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(wq_rsrc(base, (int)kOutside), dst, 16, off, step_off, 0, 0);
}
__device__ __forceinline__ void direct_load4(const char* base, wq_lptr_t dst, uint32_t off, int step_off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(wq_rsrc(base, (int)kOutside), dst, 4, off, step_off, 0, 0);
}

template <typename Policy, int TH, int NW, int WAVES, bool SB = false>
struct SkinnyCfg {
  static constexpr int KW = WAVES / NW;
  static_assert(NW * KW == WAVES && (WAVES == 4 || WAVES == 6 || WAVES == 8 || WAVES == 12), "wavefront arrangement");
  static constexpr int kRows = 8 * TH;                   // activation rows held (M <= kRows)
  static constexpr int TM = (TH + 1) / 2;                // 16-row MFMA tiles
  static_assert((2 * TH) % NW == 0, "the slab loads divide among the wavefronts of one kw");
  static constexpr int kSlabBytes = kRows * 256;         // rows x 128 k
  static constexpr int kXBytes = KW * kSlabBytes;
  static constexpr int kWBytes = WAVES * Policy::kPieces * 1024;
  static constexpr bool kStepScale = Policy::kScaleDma && !SB;  // a scale load per lane and step
  static constexpr int kStageBytes = kXBytes + kWBytes + (kStepScale ? WAVES * 256 : 0);
  static constexpr int kXLoads = 2 * TH / NW;            // slab loads (4 rows each) per wavefront and step
  static constexpr int kLoadsPerStep = kXLoads + Policy::kPieces + (kStepScale ? 1 : 0);
  static constexpr int kMaxAhead = 63 / kLoadsPerStep;   // vmcnt holds 6 bits
  static constexpr int kRedBytes = WAVES * TM * 4 * 64 * 4;
  static constexpr bool kOddStart = OddStart<Policy>::value;
};

// s_waitcnt vmcnt(groups * L) for a wavefront-uniform run-time `groups` (<= 8)
template <int L>
__device__ __forceinline__ void wait_newer_groups(int groups) {
  switch (groups) {
    case 0: WQ_SK_WAITCNT_VM(0); break;
    case 1: WQ_SK_WAITCNT_VM(1 * L <= 63 ? 1 * L : 63); break;
    case 2: WQ_SK_WAITCNT_VM(2 * L <= 63 ? 2 * L : 63); break;
    case 3: WQ_SK_WAITCNT_VM(3 * L <= 63 ? 3 * L : 63); break;
    case 4: WQ_SK_WAITCNT_VM(4 * L <= 63 ? 4 * L : 63); break;
    case 5: WQ_SK_WAITCNT_VM(5 * L <= 63 ? 5 * L : 63); break;
    case 6: WQ_SK_WAITCNT_VM(6 * L <= 63 ? 6 * L : 63); break;
    case 7: WQ_SK_WAITCNT_VM(7 * L <= 63 ? 7 * L : 63); break;
    default: WQ_SK_WAITCNT_VM(8 * L <= 63 ? 8 * L : 63); break;
  }
}

template <typename Policy, typename Epilogue, int TH, int NW, int WAVES, bool SB, bool EVEN, bool WIDE>
__global__ __launch_bounds__(64 * WAVES) void skinny_gemm_kernel(
    typename Policy::Args pargs, const half_t* __restrict__ X, half_t* __restrict__ Y, Epilogue epi,
    int M, int N, int K, int stages) {
  using Cfg = SkinnyCfg<Policy, TH, NW, WAVES, SB>;
  constexpr int KW = Cfg::KW, TM = Cfg::TM, P = Policy::kPieces;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nw = wave / KW, kw = wave % KW;
  const int lj = lane & 15, kq = lane >> 4;
  const int n0 = blockIdx.x * (16 * NW);
  const int total_steps = (K + 127) >> 7;               // 128-k steps over K
  const int nsteps = (total_steps + KW - 1) / KW;       // per wavefront (the last may be partly empty)
  const int ahead = stages - 1;

  // ---- per-lane sources: buffer descriptors at the activations and at the wavefront's first column, byte offsets ----
  // slab load i of this wavefront: rows 4*li .. 4*li+3 of the slab, li = nw*kXLoads + i
  // Buffer loads, because behind a global_load_lds the compiler waits for all LDS reads wherever it waits for one, and
  // since they take 32-bit offsets and bring zeros past K by themselves.  With the operands of the next MFMAs requested
  // before the last ones are multiplied (kAhead) and the slab's order above, at 8 shapes x M = 3 .. 64, 4 formats: 6 % faster
  // on average (q4f16_1, N = 12288, K = 4096, M = 19: 17.5 -> 13.9 us; int8, N = 5120, K = 13824, M = 48: 50.4 -> 41.0).
  // int8 with 17 .. 32 rows and two wavefronts side by side loses by that: the faster the loads of a step follow one another
  // the longer they take, the more so the more rows there are (the four slab loads of a wavefront bring as many lines as rows;
  // N = 4160, K = 13824, M = 32: 27.3 us with a test for the end of the row in front of each, 29.2 without, 32.4 as buffer
  // loads).  Without the tests the weights follow behind the products there, so that a burst is two thirds as long: 26.7 us;
  // over N = 4160 .. 8192, K = 8704 .. 28672, M = 17 .. 32 7 % faster on average than with the tests, 5 % than in one burst.
  // Where K does not come out even, the tests are needed anyway and the burst is the faster one up to 24 rows (N = 8192,
  // K = 8768, M = 17: 21.0 us, with the weights behind the products 21.7).
  constexpr bool kBuffer = !WIDE && !(P == 2 && TH == 4 && NW == 2);
  constexpr bool kLateWeights = !WIDE && !kBuffer && EVEN;
  constexpr bool kAhead = kBuffer && TH >= 4;
  using Off = std::conditional_t<kBuffer, uint32_t, int64_t>;
  Off x_off[Cfg::kXLoads];
  int x_k[Cfg::kXLoads];  // first k of the chunk in step 0
#pragma unroll
  for (int i = 0; i < Cfg::kXLoads; ++i) {
    const int li = nw * Cfg::kXLoads + i;
    const int row = 4 * li + (lane >> 4);
    x_k[i] = 8 * ((lane & 15) ^ slab_swizzle(row & 15));
    x_off[i] = (Off)min(row, M - 1) * (Off)(2 * (int64_t)K) + 2 * x_k[i];
  }
  typename Policy::Lane pl, pl0;
  Policy::init(pl, pargs, min(n0 + 16 * nw + lj, N - 1), K, N);  // clamped columns are never stored
  Policy::init(pl0, pargs, min(n0 + 16 * nw, N - 1), K, N);
  const char* const w_base = Policy::w_addr(pl0, 0, 0);
  Off w_off[P];
#pragma unroll
  for (int p = 0; p < P; ++p) w_off[p] = (Off)(Policy::w_addr(pl, 32 * kq, p) - w_base);
  const char* s_base = w_base;
  Off s_off = 0;
  if constexpr (Policy::kScaleDma) {
    s_base = Policy::s_lane(pl0);
    s_off = (Off)(Policy::s_lane(pl) - s_base);
    if constexpr (Cfg::kOddStart) {  // a pair may begin in front of its column
      s_base -= 4;
      s_off += 4;
    }
  }
  // Where K does not come out even and a lane's scales lie evenly, the step goes into the scalar offset: with a test and a
  // multiplication per lane and load in its place int8 with a scale per 64 took up to 9 % longer than with 64-bit addresses
  // (N = 4096, K = 11008: M = 16 14.4 -> 13.7 us, M = 24 21.1 -> 19.9; N = 3072, K = 8768, M = 12 12.4 -> 11.3).  Where
  // K comes out even it is faster or slower by as much, depending on the shape (int8 with a scale per 64, N = 4096, K = 13824,
  // M = 24 26.9 -> 28.1 us; int4 with one, N = 8192, K = 8192, M = 24 17.3 -> 16.4).
  constexpr bool kScaleStep = Cfg::kStepScale && kBuffer && ScaleStep<Policy>::value && !EVEN;
  uint32_t s_first = 0;
  if constexpr (kScaleStep) s_first = Policy::s_rel(pl, 32 * kq);
  typename Policy::Scale s_fixed = Policy::null_scale();
  if (!Policy::kScaleDma) s_fixed = Policy::const_scale(pl);

  unsigned char* const w_area = lds + Cfg::kXBytes + wave * (P * 1024);
  unsigned char* const s_area = lds + Cfg::kXBytes + Cfg::kWBytes + wave * 256;
  // SB: all scales of the column block (K / 32 per column), as chunks of 32 per column: chunk c is
  // one load of one wavefront, lane (j, q) bringing scales 32c + 8q .. + 7 of column j
  unsigned char* const s_block = lds + stages * Cfg::kStageBytes + nw * ((((K + 1023) >> 10)) << 10);

  auto issue_slab = [&](int it, int slot) {
    const int ks = it * KW + kw;
#pragma unroll
    for (int i = 0; i < Cfg::kXLoads; ++i) {
      // past K the slab holds zeros: the weights there are exact zeros, and zero times an infinite activation is not
      const wq_lptr_t dst = (wq_lptr_t)(lds + slot * Cfg::kStageBytes + kw * Cfg::kSlabBytes + (nw * Cfg::kXLoads + i) * 1024);
      const bool in_row = EVEN || x_k[i] < K - 128 * ks;
      if constexpr (!kBuffer) {
        const char* const src = reinterpret_cast<const char*>(X) + x_off[i] + (int64_t)ks * 256;
        __builtin_amdgcn_global_load_lds((wq_gptr_t)(in_row ? src : reinterpret_cast<const char*>(&kZeroChunk)), dst, 16, 0, 0);
      } else {
        direct_load16(reinterpret_cast<const char*>(X), dst, in_row ? x_off[i] : kOutside, ks * 256);
      }
    }
  };
  auto issue_weights = [&](int it, int slot) {
    const int stage_off = slot * Cfg::kStageBytes;
    const int ks = it * KW + kw;
    const int k0 = 128 * ks + 32 * kq;             // this lane's 32 weights
    const int k0c = EVEN || k0 < K ? k0 : 0;       // past the end: any valid address (scale is zeroed)
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const wq_lptr_t dst = (wq_lptr_t)(w_area + stage_off + p * 1024);
      if constexpr (!kBuffer)
        __builtin_amdgcn_global_load_lds((wq_gptr_t)Policy::w_addr(pl, k0c, p), dst, 16, 0, 0);
      else
        direct_load16(w_base, dst, EVEN || k0 < K ? w_off[p] : kOutside, ks * Policy::kStepStride);
    }
    if constexpr (Cfg::kStepScale) {
      const wq_lptr_t dst = (wq_lptr_t)(s_area + stage_off);
      if constexpr (!kBuffer)
        __builtin_amdgcn_global_load_lds((wq_gptr_t)Policy::s_addr(pl, k0c), dst, 4, 0, 0);
      else if constexpr (kScaleStep)
        direct_load4(s_base, dst, k0 < K ? s_off + s_first : kOutside, ks * Policy::s_step(N));
      else
        direct_load4(s_base, dst, s_off + Policy::s_rel(pl, k0c), 0);
    }
  };

  float4_t acc[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) acc[i] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

  auto compute = [&](int it, int slot) {
    const int stage_off = slot * Cfg::kStageBytes;
    const unsigned char* slab = lds + stage_off + kw * Cfg::kSlabBytes;
    if constexpr (GroupSums<Policy>::value) {
      static_assert(TM == 1);
      const int k0 = 128 * (it * KW + kw);
      const int row = lj < Cfg::kRows ? lj : lj & 7;
      mul_group_sums<Policy>(acc[0], pl, w_area + stage_off, s_area + stage_off, lj, kq, live_groups(k0, K, 4), 0, [&](int g) {
        return *reinterpret_cast<const half8_t*>(slab + row * 256 + (((4 * g + kq) ^ slab_swizzle(row & 15)) << 4));
      });
      return;
    }
    const int k0 = 128 * (it * KW + kw) + 32 * kq;
    uint4_t pieces[P];
#pragma unroll
    for (int p = 0; p < P; ++p)
      pieces[p] = *reinterpret_cast<const uint4_t*>(w_area + stage_off + p * 1024 + lane * 16);
    typename Policy::Scale s = s_fixed;
    if constexpr (Cfg::kStepScale)
      s = Policy::pick_scale(pl, *reinterpret_cast<const half2_t*>(s_area + stage_off + lane * 4), kq);
    if constexpr (SB) {
      const int g = (EVEN || k0 < K ? k0 : 0) >> 5;  // chunk g / 32, fetched by lane (j, (g / 8) % 4)
      s = *reinterpret_cast<const half_t*>(s_block + (g >> 5) * 1024 + (((g >> 3) & 3) * 16 + lj) * 16 +
                                           (g & 7) * 2);
    }
    if constexpr (ColumnScale<Policy>::value) {
      if (!EVEN && k0 >= K) zero_codes<Policy>(pieces);
    } else {
      if (!EVEN && k0 >= K) s = Policy::null_scale();  // code * 0 = exact zero for the weights past K
    }
    half8_t bop[4];
    Policy::dequant(pieces, s, bop);
    // rows past the slab (M <= 8 uses half a tile) re-read a held row: never stored
    auto a_operand = [&](int t, int i) {
      const int row = (16 * i + lj < Cfg::kRows) ? 16 * i + lj : 16 * i + (lj & 7);
      return *reinterpret_cast<const half8_t*>(slab + row * 256 + (((4 * kq + t) ^ slab_swizzle(row & 15)) << 4));
    };
    if constexpr (kAhead) {
      half8_t aop[2][TM];
#pragma unroll
      for (int i = 0; i < TM; ++i) aop[0][i] = a_operand(0, i);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (t < 3) {
#pragma unroll
          for (int i = 0; i < TM; ++i) aop[(t + 1) & 1][i] = a_operand(t + 1, i);
        }
        __builtin_amdgcn_sched_barrier(0x6);  // only the unpacking may move past
#pragma unroll
        for (int i = 0; i < TM; ++i)
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(aop[t & 1][i], bop[t], acc[i], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0x6);
      }
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_operand(t, i), bop[t], acc[i], 0, 0, 0);
      }
    }
  };

  // ---- prologue: the scale block (its loads are older than every step's, so each wavefront's
  // part has landed when its first wait returns; the barrier of step 0 covers the others'), then
  // fill the ring ----
  if constexpr (SB) {
    for (int c = kw; c * 1024 < K; c += KW) {
      const int g = 32 * c + 8 * kq;
      direct_load16(s_base, (wq_lptr_t)(s_block + c * 1024), s_off + (g * 32 < K ? g : 0) * 2, 0);
    }
  }
  auto fill = [&](int p) {
    issue_slab(p, p);
    issue_weights(p, p);
  };
  if constexpr (TH <= 2) {
    // one or two rounds; unrolled by eight, what the compiler computes in front of them delays the first load (N = K = 1024,
    // up to 16 rows: 3.6 .. 3.9 -> 3.4 .. 3.7 us, what they took with addresses of 64 bits)
#pragma unroll 1
    for (int p = 0; p < ahead && p < nsteps; ++p) fill(p);
  } else {
    for (int p = 0; p < ahead && p < nsteps; ++p) fill(p);
  }
  int cslot = 0;                       // slot of the step being computed
  int islot = ahead;                   // slot the next issue goes to
  for (int it = 0; it < nsteps; ++it) {
    wait_newer_groups<Cfg::kLoadsPerStep>(min(ahead - 1, nsteps - 1 - it));  // steps issued after step `it`
    if (NW > 1 || (SB && KW > 1 && it == 0)) __builtin_amdgcn_s_barrier();
    // the slot refilled now was computed in the previous iteration (by everyone: barrier above)
    if (it + ahead < nsteps) {
      issue_slab(it + ahead, islot);
      if constexpr (!kLateWeights) {
        issue_weights(it + ahead, islot);
        islot = islot + 1 == stages ? 0 : islot + 1;
      }
    }
    compute(it, cslot);
    if constexpr (kLateWeights) {
      if (it + ahead < nsteps) {
        issue_weights(it + ahead, islot);
        islot = islot + 1 == stages ? 0 : islot + 1;
      }
    }
    cslot = cslot + 1 == stages ? 0 : cslot + 1;
  }

  // ---- reduce the KW partial sums of each column block through LDS, then store ----
  if (KW > 1) {
    __syncthreads();  // all ring slots idle
    float* red = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[((wave * TM + i) * 4 + r) * 64 + lane] = acc[i][r];
    __syncthreads();
    if (kw == 0) {
#pragma unroll
      for (int o = 1; o < KW; ++o)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[i][r] += red[(((wave + o) * TM + i) * 4 + r) * 64 + lane];
    }
  }
  if (kw == 0) {
    const int col = n0 + 16 * nw + lj;
    if (col < N) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = 16 * i + 4 * kq + r;
          float v = acc[i][r];
          if constexpr (ColumnScale<Policy>::value) v *= (float)s_fixed;
          if (m < M) Y[(int64_t)m * N + col] = epi(v, m, col);
        }
    }
  }
}


constexpr int kSkinnyLdsBudget = 156 * 1024;  // of the 160 KB of a CU

// ---------------------------------------------------------------------------------
// M <= 16: the activations stay in registers.
//
// The ring kernel above re-reads the activations once per workgroup and keeps two thirds
// of its loads in flight on those slabs; loads retire in order, so its weight stream is
// only as deep as the slab ring.  For one 16-row tile the activations fit the register
// file instead: a workgroup's WAVES wavefronts split K into contiguous runs of NSTEP
// steps of 128 k, and wavefront w keeps the MFMA A operands of its run (16 rows x
// 128*NSTEP k: 16*NSTEP registers) for the whole kernel.  The workgroups are persistent
// (one per CU) and walk over 16-column tiles; the only loads inside the walk are the
// codes and scales, through a wavefront-private ring in LDS that runs kDepth steps ahead
// (across tiles).  Per tile the WAVES partial sums meet in LDS and one wavefront (taking
// turns) adds them and stores.  Measured: with loads only it streams 2 TB/s however
// deep the ring (and no more from sixteen wavefronts than from eight), so it wins where
// the ring kernel pays most for the slabs (K = 8192, many tiles per CU) and loses at
// K = 4096.
//
// Every policy hands its scale over as a 4-byte pair per lane and step here
// (Policy::s_pair_addr), so that the walk has no load the compiler must wait for.
template <typename Policy, int NSTEP, int WAVES>
struct XregCfg {
  static constexpr int kStepBytes = Policy::kPieces * 1024 + 256;
  static constexpr int kLoadsPerStep = Policy::kPieces + 1;
  static constexpr int kRedBytes = 2 * WAVES * 1024;
  static constexpr int kFit = (kSkinnyLdsBudget - kRedBytes) / (WAVES * kStepBytes);
  static constexpr int kCount = 63 / kLoadsPerStep + 1;  // vmcnt holds 6 bits
  static constexpr int kWant = 3 * NSTEP;
  static constexpr int kDepth = kFit < kCount ? (kFit < kWant ? kFit : kWant) : (kCount < kWant ? kCount : kWant);
  static_assert(kDepth >= 2, "ring too small");
  static constexpr int kLdsBytes = WAVES * kDepth * kStepBytes + kRedBytes;
};

template <typename Policy, typename Epilogue, int NSTEP, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void skinny_xreg_kernel(
    typename Policy::Args pargs, const half_t* __restrict__ X, half_t* __restrict__ Y, Epilogue epi,
    int M, int N, int K) {
  using Cfg = XregCfg<Policy, NSTEP, WAVES>;
  constexpr int P = Policy::kPieces, L = Cfg::kLoadsPerStep, D = Cfg::kDepth;
  constexpr int QA = D / NSTEP;  // the step D ahead of step s is step (s + D) % NSTEP, QA or QA + 1 tiles ahead
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lj = lane & 15, kq = lane >> 4;
  const int tiles = (N + 15) >> 4;
  const int grid = gridDim.x;
  unsigned char* const ring = lds + wave * (D * Cfg::kStepBytes);
  float4_t* const red = reinterpret_cast<float4_t*>(lds + WAVES * D * Cfg::kStepBytes);

  // ---- the A operands of this wavefront's run of K (zero past M and past K) ----
  half8_t a[NSTEP][4];
  int k0c[NSTEP];  // this lane's 32 weights of step s (any valid k when past K)
  bool past[NSTEP];  // past K: the scale is zeroed too, the one fetched may be another row's and 0 * inf is not 0
#pragma unroll
  for (int s = 0; s < NSTEP; ++s) {
    const int k0 = (wave * NSTEP + s) * 128 + 32 * kq;
    const bool held = lj < M && k0 < K;
    past[s] = k0 >= K;
    k0c[s] = past[s] ? 0 : k0;
    if constexpr (GroupSums<Policy>::value) {  // operand t: k 8kq .. + 7 of group t
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int kt = (wave * NSTEP + s) * 128 + 32 * t;
        const bool held_t = lj < M && kt < K;
        const half8_t v = *reinterpret_cast<const half8_t*>(held_t ? X + (int64_t)lj * K + kt + 8 * kq : X);
        a[s][t] = held_t ? v : half8_t{};
      }
      continue;
    }
    const half_t* src = held ? X + (int64_t)lj * K + k0 : X;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const half8_t v = *reinterpret_cast<const half8_t*>(src + 8 * t);
      a[s][t] = held ? v : half8_t{};
    }
  }

  // lane state of the tiles QA and QA + 1 tiles ahead (whose loads are being issued)
  typename Policy::Lane pl[2];
  bool valid[2] = {false, false};
  auto set_tile = [&](int which, int tile) {
    valid[which] = tile < tiles;  // past the end: every lane re-reads one address
    Policy::init(pl[which], pargs, min(min(tile, tiles - 1) * 16 + lj, N - 1), K, N);
  };
  auto issue = [&](int which, int s, int slot) {
    unsigned char* dst = ring + slot * Cfg::kStepBytes;
#pragma unroll
    for (int p = 0; p < P; ++p)
      __builtin_amdgcn_global_load_lds(
          (wq_gptr_t)(valid[which] ? Policy::w_addr(pl[which], k0c[s], p) : reinterpret_cast<const char*>(X)),
          (wq_lptr_t)(dst + p * 1024), 16, 0, 0);
    __builtin_amdgcn_global_load_lds(
        (wq_gptr_t)(valid[which] ? Policy::s_pair_addr(pl[which], k0c[s]) : reinterpret_cast<const char*>(X)),
        (wq_lptr_t)(dst + P * 1024), 4, 0, 0);
  };

  // ---- prologue: the first D steps (slot = flat step % D) ----
#pragma unroll
  for (int f = 0; f < D; ++f) {
    if (f % NSTEP == 0) set_tile(0, blockIdx.x + (f / NSTEP) * grid);
    issue(0, f % NSTEP, f);
  }
  // the activations are in registers before the walk starts
#pragma unroll
  for (int s = 0; s < NSTEP; ++s)
#pragma unroll
    for (int t = 0; t < 4; ++t) asm volatile("" : "+v"(a[s][t]));
  typename Policy::Lane pl0;  // for pick_scale, which depends on the lane only
  Policy::init(pl0, pargs, min(blockIdx.x * 16 + lj, N - 1), K, N);
  set_tile(0, blockIdx.x + QA * grid);

  int slot = 0;  // of step 0 of the current tile
  int turn = 0;
  uint32_t run_groups = 0;  // the 32-k groups of this wavefront's run that exist (GroupSums)
  if constexpr (GroupSums<Policy>::value) run_groups = live_groups(wave * NSTEP * 128, K, 4 * NSTEP);
  for (int tile = blockIdx.x; tile < tiles; tile += grid) {
    set_tile(1, tile + (QA + 1) * grid);
    if constexpr (GroupSums<Policy>::value) asm volatile("" : "+v"(run_groups));  // or a mask per group is kept: they spill
    const uint32_t live = __builtin_amdgcn_readfirstlane(run_groups);
    float4_t acc = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    float column_scale = 0.0f;
#pragma unroll
    for (int s = 0; s < NSTEP; ++s) {
      WQ_SK_WAITCNT_VM((D - 1) * L);  // issued after this step's loads: the D - 1 steps that follow it
      int sl = slot + s;
      if (sl >= D) sl -= D;
      const unsigned char* src = ring + sl * Cfg::kStepBytes;
      if constexpr (GroupSums<Policy>::value) {
        mul_group_sums<Policy>(acc, pl0, src, src + P * 1024, lj, kq, live, 4 * s, [&](int g) { return a[s][g]; });
        asm volatile("" : "+v"(acc));  // scaled in every step: left to the end of the tile the sums of all steps spill
      } else {
        uint4_t pieces[P];
#pragma unroll
        for (int p = 0; p < P; ++p) pieces[p] = *reinterpret_cast<const uint4_t*>(src + p * 1024 + lane * 16);
        const half2_t pair = *reinterpret_cast<const half2_t*>(src + P * 1024 + lane * 4);
        typename Policy::Scale scale = Policy::pick_scale(pl0, pair, kq);
        if constexpr (ColumnScale<Policy>::value) {
          if (past[s]) zero_codes<Policy>(pieces);
          column_scale = (float)scale;
        } else {
          if (past[s]) scale = Policy::null_scale();
        }
        half8_t bop[4];
        Policy::dequant(pieces, scale, bop);
#pragma unroll
        for (int t = 0; t < 4; ++t) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[s][t], bop[t], acc, 0, 0, 0);
      }
      // the slot is free once its contents are in registers; it takes the step D ahead
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      issue((s + D) / NSTEP - QA, (s + D) % NSTEP, sl);
    }
    slot = (slot + NSTEP) % D;
    pl[0] = pl[1];
    valid[0] = valid[1];

    // ---- the WAVES partial sums of the tile meet in LDS (two buffers, by turns) ----
    float4_t* const buf = red + (turn & 1) * (WAVES * 64);
    if constexpr (ColumnScale<Policy>::value) {
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] *= column_scale;
    }
    buf[wave * 64 + lane] = acc;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (wave == turn % WAVES) {
      float4_t sum = buf[lane];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) {
        const float4_t v = buf[w * 64 + lane];
        sum[0] += v[0]; sum[1] += v[1]; sum[2] += v[2]; sum[3] += v[3];
      }
      const int col = tile * 16 + lj;
      if (col < N) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = 4 * kq + r;
          if (m < M) Y[(int64_t)m * N + col] = epi(sum[r], m, col);
        }
      }
    }
    ++turn;
  }
  WQ_SK_WAITCNT_VM(0);  // the loads past the last tile land before the LDS is given back
}

template <typename Policy, typename Epilogue, int NSTEP, int WAVES>
static int launch_xreg(const char* who, const typename Policy::Args& pargs, const uint16_t* x, uint16_t* y,
                       const Epilogue& epi, int64_t M, int64_t N, int64_t K, hipStream_t stream) {
  using Cfg = XregCfg<Policy, NSTEP, WAVES>;
  auto kern = skinny_xreg_kernel<Policy, Epilogue, NSTEP, WAVES>;
  const int64_t tiles = (N + 15) / 16;
  const int64_t blocks = tiles < cu_count() ? tiles : cu_count();
  static DynamicLdsLimit limit;  // per instantiation
  WQ_HIP(limit.ensure(reinterpret_cast<const void*>(kern), 160 * 1024));
  WQ_LAUNCH(who, kern, dim3((unsigned)blocks), dim3(64 * WAVES), Cfg::kLdsBytes, stream, pargs,
            (const half_t*)x, (half_t*)y, epi, (int)M, (int)N, (int)K);
  tuning().small_batch_form = kXregForm;
  return WQ_OK;
}

// K up to 64 steps of 128 (8192) is held by 8 wavefronts x 4 or 8 steps (64 or 128 registers;
// 11 steps for K = 11008 spill)
inline bool xreg_fits(int64_t M, int64_t K) { return M <= 16 && K <= 64 * 128; }

template <typename Policy, typename Epilogue>
static int launch_xreg_auto(const char* who, const typename Policy::Args& pargs, const uint16_t* x,
                            uint16_t* y, const Epilogue& epi, int64_t M, int64_t N, int64_t K,
                            hipStream_t stream) {
  const int64_t steps = (K + 127) / 128;
  if (steps <= 32) return launch_xreg<Policy, Epilogue, 4, 8>(who, pargs, x, y, epi, M, N, K, stream);
  return launch_xreg<Policy, Epilogue, 8, 8>(who, pargs, x, y, epi, M, N, K, stream);
}

// overrides for tests and measurement (tuning.h; 0 = automatic)
// waves: 1 = the ring kernel (12: with twelve wavefronts, nw = 3), 2 = the kernel that holds the activations in registers (where it fits)
struct SkinnyTuning {
  int nw, stages, waves;
};
inline SkinnyTuning skinny_tuning() {
  const Tuning& t = tuning();
  return SkinnyTuning{t.skinny_nw, t.skinny_stages, t.skinny_waves};
}

template <typename Policy, typename Epilogue, int TH, int NW, int WAVES, bool SB, bool EVEN, bool WIDE = false>
static int launch_skinny_form(const char* who, const typename Policy::Args& pargs, const uint16_t* x, uint16_t* y,
                              const Epilogue& epi, int64_t M, int64_t N, int64_t K, int want_stages,
                              hipStream_t stream) {
  // one fetch of all scales where the policy allows it and the block is small (two column
  // blocks at most: more would cost a workgroup per CU)
  if constexpr (!SB && !WIDE && Policy::kCanScaleBlock && NW <= 2) {
    if (K <= kScaleBlockMaxK && Policy::scale_block_ok(pargs, K) &&
        2 * SkinnyCfg<Policy, TH, NW, WAVES, true>::kStageBytes + NW * scale_block_stride((int)K) <=
            kSkinnyLdsBudget)
      return launch_skinny_form<Policy, Epilogue, TH, NW, WAVES, true, EVEN>(who, pargs, x, y, epi, M, N, K,
                                                                             want_stages, stream);
  }
  using Cfg = SkinnyCfg<Policy, TH, NW, WAVES, SB>;
  auto kern = skinny_gemm_kernel<Policy, Epilogue, TH, NW, WAVES, SB, EVEN, WIDE>;
  const int64_t blocks = (N + 16 * NW - 1) / (16 * NW);
  int stages = want_stages;
  if (stages > Cfg::kMaxAhead + 1) stages = Cfg::kMaxAhead + 1;
  if (stages > 9) stages = 9;
  const int sblock_bytes = SB ? NW * scale_block_stride((int)K) : 0;  // after the ring
  if (stages * Cfg::kStageBytes + sblock_bytes > kSkinnyLdsBudget)
    stages = (kSkinnyLdsBudget - sblock_bytes) / Cfg::kStageBytes;
  WQ_REQUIRE(stages >= 2, "%s: internal: no room for a 2-slot ring", who);
  int lds_bytes = stages * Cfg::kStageBytes + sblock_bytes;
  if (lds_bytes < Cfg::kRedBytes) lds_bytes = Cfg::kRedBytes;
  static DynamicLdsLimit limit;  // per instantiation
  WQ_HIP(limit.ensure(reinterpret_cast<const void*>(kern), 160 * 1024));
  WQ_LAUNCH(who, kern, dim3((unsigned)blocks), dim3(64 * WAVES), lds_bytes, stream, pargs,
            (const half_t*)x, (half_t*)y, epi, (int)M, (int)N, (int)K, stages);
  tuning().small_batch_form = small_batch_form(TH, NW, WAVES);
  return WQ_OK;
}

// EVEN: K is whole steps for every wavefront (K % (128 * KW) == 0), so that nothing lies past it.
template <typename Policy, typename Epilogue, int TH, int NW, int WAVES>
static int launch_skinny(const char* who, const typename Policy::Args& pargs, const uint16_t* x, uint16_t* y,
                         const Epilogue& epi, int64_t M, int64_t N, int64_t K, int want_stages,
                         hipStream_t stream) {
  if constexpr (!GroupSums<Policy>::value) {  // (those are for K % 64 == 32)
    if (K % (128 * (WAVES / NW)) == 0)
      return launch_skinny_form<Policy, Epilogue, TH, NW, WAVES, false, true>(who, pargs, x, y, epi, M, N, K,
                                                                              want_stages, stream);
  }
  return launch_skinny_form<Policy, Epilogue, TH, NW, WAVES, false, false>(who, pargs, x, y, epi, M, N, K,
                                                                           want_stages, stream);
}

// Picks the arrangement from the shape (timings of the Llama-7B layer shapes): few
// columns per workgroup while the matrix is small, so that every CU gets work; more
// columns per workgroup for tall matrices and larger M, where the re-reads of the
// activations (once per workgroup) would otherwise outweigh the weight stream.
template <typename Policy, typename Epilogue>
static int launch_skinny_auto(const char* who, const typename Policy::Args& pargs, const uint16_t* x,
                              uint16_t* y, const Epilogue& epi, int64_t M, int64_t N, int64_t K,
                              hipStream_t stream) {
  const SkinnyTuning t = skinny_tuning();
  // activations in registers where that kernel is the faster one: 4096 < K <= 8192 and at least
  // four column tiles per CU (N = 28672, K = 8192, int8, M = 4: 60 -> 48 us; with two tiles per CU, or at
  // K = 4096, the ring kernel is the faster one)
  if constexpr (UsesXreg<Policy>::value) {
    if (xreg_fits(M, K) && Policy::pair_aligned(pargs) && (t.waves == 2 || (t.waves == 0 && K > 4096 && N / 16 >= 4 * (int64_t)cu_count())))
      return launch_xreg_auto<Policy, Epilogue>(who, pargs, x, y, epi, M, N, K, stream);
  }
  if (K >= kSkinnyMaxK || Policy::s_reach(pargs, N, K) >= (int64_t)kOutside)  // (four wavefronts, two ring slots)
    return launch_skinny_form<Policy, Epilogue, GroupSums<Policy>::value ? 1 : 8, 1, 4, false, false, true>(who, pargs, x, y, epi, M, N, K, 2, stream);
  const int64_t per_cu = (N / 16) / cu_count();
  int nw = 1;
  if (per_cu >= 2) nw = M <= 8 ? (per_cu >= 4 ? 2 : 1) : M <= 16 ? 2 : 4;
  // wide matrices and more than 16 rows: all eight wavefronts side by side (128 columns per
  // workgroup, each wavefront the whole K), which halves the re-reads of x again, as long as
  // most CUs still get a workgroup (int8, K = 8192, N = 28672, M = 64: 80 -> 62 us)
  if (M > 16 && N / 128 >= (cu_count() * 5) / 8) nw = 8;
  // ... corrected for how the workgroups fill the machine.  A workgroup of nw wavefronts takes nw column tiles
  // and stages the activations once, which costs about as much as one tile (two from 33 rows on): the launch
  // lasts about (rounds of the CUs) x (nw + that).  Fewer wavefronts side by side where that is shorter
  // (N = 8192 with 4: 128 workgroups on 256 CUs; K = 28672, M = 32: 102 -> 62 us), two instead of one where
  // one leaves a second, partly filled round (N = 5120, K = 13824, M = 32: 43 -> 31 us; N = 6144, K = 4096,
  // M = 64: 22 -> 14 us).  Up to 8 rows the choice above stands (measured either way).
  if (M > 8 && !t.nw) {
    const int64_t tiles = (N + 15) / 16, cus = cu_count();
    const double cx = M > 32 ? 2.0 : 1.0;
    auto cost = [&](int w) { return (double)((tiles + w * cus - 1) / (w * cus)) * (w + cx); };
    while (nw > 1 && cost(nw / 2) < cost(nw) - 1e-9) nw /= 2;
    if (nw == 1 && cost(2) < cost(1) - 1e-9) nw = 2;
  }
  // 17 .. 24 rows: slabs of 24 rows and three wavefronts side by side where four or eight leave a second, partly filled
  // round: between four and six tiles per CU in every format (M = 19, q4f16_1 / int8: N = 18432, K = 4096 28.8 -> 20.0 /
  // 32.3 -> 20.4 us, N = 24576, K = 6144 36.7 -> 30.8 / 40.1 -> 35.1; N = 16384 and N = 24640 lose 10 .. 30 %), and between
  // two and three, where it makes one whole round.  There the one workgroup that a CU has takes twelve wavefronts, four
  // along K: with six the matrix cores wait for the unpacking.  M = 19, weights from memory, q4f16_1 with four side by
  // side / int8 with three and six / int4 with four -> twelve: N = 12288, K = 4096 13.9 / 14.5 / 13.6 -> 12.4 / 14.2 / 11.7 us,
  // K = 13824 39.0 / 37.2 / 36.3 -> 32.2 / 35.7 / 27.7; N = 8256 (the first width), K = 8192 24.0 / 22.9 / 23.0 -> 19.8 / 20.0 / 17.7.
  // Below K = 2048 a step or two per wavefront is too little (K = 1056 6.5 -> 6.7; int8, K = 1024 6.7 -> 7.1).  Between four
  // and six tiles per CU it loses (N = 22016, K = 4096 20.5 -> 21.2).
  bool twelve = false;
  if (M > 16 && M <= 24) {
    const int64_t tiles = (N + 15) / 16, cus = cu_count();
    const bool one_round = tiles > 2 * cus && tiles <= 3 * cus;
    twelve = one_round && K >= 2048;
    if ((tiles > 4 * cus && tiles <= 6 * cus) || twelve || (one_round && Policy::kPieces == 2)) nw = 3;
  }
  if (t.nw) nw = t.nw, twelve = t.waves == 12;
  if (nw == 3 && (M <= 16 || M > 24)) nw = 4;
  if (M <= 8 && nw >= 4) nw = 2;  // 8 rows are two slab loads: at most two wavefronts share them
  // three ring slots for four or more wavefronts side by side, and for two when every workgroup has a CU of
  // its own anyway (N = 8192, K = 28672, M = 16: 67 -> 46 us; with more workgroups than CUs the third slot
  // costs a resident workgroup: N = 10240, K = 8192, M = 16: 20.9 -> 27.4 us)
  const int64_t wgs = ((N + 15) / 16 + nw - 1) / nw;
  const int stages = t.stages ? t.stages : (nw >= 4 || (nw >= 2 && M > 8 && wgs <= cu_count()) ? 3 : 2);
  // eight wavefronts where two ring slots of that arrangement fit LDS, else four
#define WQ_SK_GO(TH, NW, WAVES)                                                                        \
  do {                                                                                                 \
    if constexpr (2 * SkinnyCfg<Policy, TH, NW, WAVES>::kStageBytes <= kSkinnyLdsBudget)               \
      return launch_skinny<Policy, Epilogue, TH, NW, WAVES>(who, pargs, x, y, epi, M, N, K, stages,    \
                                                            stream);                                   \
    else                                                                                               \
      return launch_skinny<Policy, Epilogue, TH, NW, 4>(who, pargs, x, y, epi, M, N, K, stages,        \
                                                        stream);                                       \
  } while (0)
  if (M <= 8) {
    if (nw == 2) WQ_SK_GO(1, 2, 8);
    WQ_SK_GO(1, 1, 8);
  }
  if constexpr (GroupSums<Policy>::value) {
    return fail(WQ_EINVAL, "%s: internal: more than 8 rows", who);
  } else {
  if (M <= 16 && nw != 8) {
    if (nw == 4) WQ_SK_GO(2, 4, 8);
    if (nw == 2) WQ_SK_GO(2, 2, 8);
    WQ_SK_GO(2, 1, 8);
  }
  if (nw == 3) {
    if (twelve) WQ_SK_GO(3, 3, 12);
    WQ_SK_GO(3, 3, 6);
  }
  // slabs of 24 rows also for int8 with one column block (M = 17 / 24, before -> now, weights from memory: N = 2048, K = 4096, a scale per
  // 64 7.6 / 8.0 -> 6.0 / 6.8 us; N = 4096, K = 11008 21.4 / 21.9 -> 16.7 / 18.5; per column, K = 13824, M = 20 22.0 -> 19.7; K = 1088
  // 5.1 / 5.5 -> 5.0 / 5.6).  int4 and AutoGPTQ gain 2 .. 4 %, q4f16_1 between 2 and -4 %.
  if constexpr (Policy::kPieces == 2) {
    if (M <= 24 && nw == 1 && K >= 2048) WQ_SK_GO(3, 1, 8);
  }
  if (M <= 32) {
    if (nw == 8) WQ_SK_GO(4, 8, 8);
    if (nw == 4) WQ_SK_GO(4, 4, 8);
    if (nw == 2) WQ_SK_GO(4, 2, 8);
    WQ_SK_GO(4, 1, 8);
  }
  // 33 .. 48 rows: slabs of 48, a quarter less to bring and to multiply (M = 40, before -> now, weights from memory: N = K = 4096
  // q4f16_1 9.7 -> 9.1 us, int8 12.1 -> 11.5, int4 10.0 -> 9.3; N = K = 8192 q4f16_1 28.8 -> 23.8; N = 12288, K = 4096 18.2 -> 16.9,
  // 18.3 -> 17.3, 16.8 -> 14.6; N = 16384, K = 13824 55.6 -> 51.3, 57.5 -> 54.4, 48.4 -> 42.1).  Not with eight column blocks (the
  // twelve loads of a slab do not divide among them), and for int8 not with two (N = 8192, K = 4096, M = 40 14.4 -> 16.7) and
  // with four up to 40 rows (a scale per 64, N = 11008, K = 11008, M = 33 42.9 -> 40.1, M = 48 45.4 -> 47.0);
  // with two otherwise up to 40 rows, or above K = 4096 (int4 with a scale per 64, N = 6144, M = 36 / 48: K = 4096 13.3 / 13.3 -> 12.5 / 13.9,
  // K = 5120 17.5 / 18.6 -> 16.6 / 17.8).
  if (M <= 48 && nw <= 4) {
    if constexpr (Policy::kPieces == 1) {
      if (nw == 2 && (M <= 40 || K > 4096)) WQ_SK_GO(6, 2, 8);
    }
    if (nw == 4 && (Policy::kPieces == 1 || M <= 40)) WQ_SK_GO(6, 4, 8);
    if (nw == 1) WQ_SK_GO(6, 1, 8);
  }
  if (nw == 8) WQ_SK_GO(8, 8, 8);
  if (nw == 4) WQ_SK_GO(8, 4, 8);
  if (nw == 2) WQ_SK_GO(8, 2, 8);
  WQ_SK_GO(8, 1, 8);
  }
#undef WQ_SK_GO
}

}  // namespace wq
#endif  // RELAX_AMD_CSRC_SKINNY_GEMM_H_
