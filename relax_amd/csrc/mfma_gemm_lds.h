// Prefill GEMM, fully LDS-staged variant for the gfx950 matrix cores, both weight formats:
//   y[m,n] = epilogue( sum_k x[m,k] * dequant(w)[n,k] )
//
// Every operand of a K-step (64 k) travels global -> LDS with direct loads: no staging registers, no VALU work, and the
// loads of the next two or more steps are in flight while a step is multiplied (a ring of 3 slots, or of up to 6
// where one workgroup per CU leaves room in LDS; what pays is a 4-slot ring under 256 x 128 tiles).  Per slot:
//   A   BM rows x 128 B of activations, 16-byte chunk c of row r at slot position
//       c ^ ((r >> 1) & 7) (the swizzle is applied to the GLOBAL address each lane fetches,
//       because the LDS side of a direct load is fixed: lane l writes 16 bytes at
//       base + 16*l);
//   B   BN columns x 32 or 64 B of packed codes, still packed, in the order the weight
//       format's policy fetches them;
//   S   (formats with a scale per group) BN x 4 B: the two scales of the step, or the pair of a group; BN x 8 B where
//       the two scales straddle aligned words (format A, K % 64 == 32).
// A wavefront then reads, per K-step, TM*4 activation fragments, and per weight
// sub-tile its 32 codes (16 or 32 bytes) plus one scale: MFMA lane (j, h) needs 8
// K-values of column j per MFMA, so the weights are dequantized in registers by the
// policy's bit-exact pair function (natural K order, hence no rearrangement of the
// activations) and never exist in LDS as fp16.
//
// Synchronisation: vector memory operations retire in order, so s_waitcnt vmcnt(loads of
// one step) means "this wavefront's loads of the step before have landed"; one raw
// s_barrier per K-step then says the same for the whole workgroup (the fence in
// __syncthreads would force vmcnt(0)).  The schedule inside a K-step is described at
// gemm_lds_tile.
//
// A weight policy provides
//   kColBytes            packed bytes per column and K-step (32 or 64)
//   kScaleBytes          bytes of scales per column and K-step staged in LDS (0, 4, or 8 as two planes of 4)
//   Args, Frag, Scale    kernel arguments; a lane's packed codes of one column for one step; what
//                        pair() needs besides the codes (the scale, with the zero point where the format has one)
//   b_src(args, n0, q, N, K)   global address (step 0) of 16-byte chunk q of the B tile at column n0
//   kStepStride          bytes between consecutive K-steps of a chunk
//   s_src(args, n, K)    global address (step 0) of the 4 scale bytes of column n       (kScaleBytes > 0)
//   s_offset(args, ks)   byte offset of step ks from there                              (kScaleBytes > 0)
//   read_scale(p, lh)    Scale from the 4 staged bytes of a column, for lane half lh    (kScaleBytes > 0)
//   s_src2(args, n, K)   the same for the second plane                                  (kScaleBytes == 8)
//   read_scale2(p, plane, n, lh)   Scale from the 4 staged bytes of column n at p and those at p + plane
//                                                                                       (kScaleBytes == 8)
//   const_scale(args, n) the Scale of column n                                          (kScaleBytes == 0)
//   read(frag, bslot, n_local, lh)   LDS -> registers
//   pair(frag, kk, j, scale)   dequantized weights (k = 8kk + 2j, 8kk + 2j + 1) of the lane's column,
//                              = pair_finish(pair_bits(frag, kk, j), scale): the two exact fp16 integers as a bit
//                              pattern, the offset of the codes subtracted where it is known beforehand, then
//                              times the scale (after the zero point, where there is one).  The K loop runs the
//                              two halves in different MFMA slots: the whole chain does not fit behind one MFMA.
// and, only where the scale of a weight depends on its k inside the step (scales along N):
//   phase_begin(scale, kk)     called once per column sub-tile in front of the phase that unpacks the weights
//                              of MFMA kk: fetches what pair_finish_at needs for them
//   pair_finish_at(bits, scale, j)   pair_finish for pair j of that MFMA
// and, only where K may end with half a step (K % 64 == 32):
//   half_step(args, n, k0, K, lh, out[2])   the weights k0 + 16c + 8lh .. + 7 of column n, c = 0, 1
#ifndef RELAX_AMD_CSRC_MFMA_GEMM_LDS_H_
#define RELAX_AMD_CSRC_MFMA_GEMM_LDS_H_

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "gemm_epilogue.h"
#include "tuning.h"
#include "wq_device.h"
#include "wq_host.h"

namespace wq {

// Policy::kRegB = true: weights and scales go from memory to registers (gemm_rb_tile).
template <class P, class = void>
struct RegB : std::false_type {};
template <class P>
struct RegB<P, std::void_t<decltype(P::kRegB)>> : std::bool_constant<P::kRegB> {};

template <class Policy, int TM, int TN, int WM, int WN, int WPE>
struct LdsGemmCfg {
  static_assert(WM * WN == 4, "four wavefronts per workgroup");
  static constexpr int kThreads = 256;
  static constexpr int BM = 32 * TM * WM;
  static constexpr int BN = 32 * TN * WN;
  static constexpr int kAOff = 0;
  static constexpr int kBOff = BM * 128;
  static constexpr int kSOff = kBOff + BN * Policy::kColBytes;
  static constexpr int kStageBytes = RegB<Policy>::value ? kBOff : kSOff + BN * Policy::kScaleBytes;
  // ring slots: loads of kStages - 1 steps are in flight while a step is multiplied; four where a
  // single workgroup per CU leaves room for them in the 160 KiB of LDS
  static constexpr int kFit = (158 * 1024) / kStageBytes;
  static constexpr int kStages = RegB<Policy>::value ? 4 : WPE == 1 ? (kFit >= 6 ? 6 : kFit >= 4 ? kFit : 3) : 3;
  static constexpr int kLdsBytes = kStages * kStageBytes;
  static constexpr int kALoads = BM / 32;   // direct loads per wavefront per step (64 chunks each)
  static constexpr int kBLoads = BN * Policy::kColBytes / 4096;
  static_assert(BN % 128 == 0 && BN <= 256, "B tile: 128 or 256 columns");
  static constexpr int kSLoads = Policy::kScaleBytes / 4;
  static constexpr int kLoadsPerStage = kALoads + kBLoads + kSLoads;
};

// XOR pattern of the activation tile: consecutive rows alternate between the two
// 128-byte halves of the bank space, so pairs of rows share one pattern value.
#define WQ_SWZ(r) (((r) >> 1) & 7)
#define WQ_WAITCNT_VM(n) __builtin_amdgcn_s_waitcnt(((n)&0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0xF << 8))
// the same with lgkmcnt(0): this wavefront's LDS reads have returned as well
#define WQ_WAITCNT_VM_LGKM0(n) __builtin_amdgcn_s_waitcnt(((n)&0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0x0 << 8))

template <class P, class = void>
struct ScalePerK : std::false_type {};
template <class P>
struct ScalePerK<P, std::void_t<decltype(&P::phase_begin)>> : std::true_type {};

template <class P, class = void>
struct HalfStep : std::false_type {};
template <class P>
struct HalfStep<P, std::void_t<decltype(&P::half_step)>> : std::true_type {};

// Policy::kColumnScale = true (kScaleBytes == 0): the sums take the column's scale, pair_finish gives the codes as they are.

// Policy::kWide = true: 64-bit addresses, for a K whose byte offsets inside a tile do not fit 32 bits.
template <class P, class = void>
struct Wide : std::false_type {};
template <class P>
struct Wide<P, std::void_t<decltype(P::kWide)>> : std::bool_constant<P::kWide> {};
// ... which they do below this one (256 rows of activations)
constexpr int64_t kLdsGemmMaxK = 1 << 23;

// What follows the K loop: the sums of the two sets of wavefronts (KW = 2), then the epilogue.  Both stage in the ring, so
// it has to be idle: no direct load of any wavefront on its way, loads past the last step included, and a barrier behind
// the wait for them.  Both tile bodies end with that (check_ring_asm.py refuses a build without it).
template <class Policy, class Epilogue, int TM, int TN, int WM, int WN, int WPE, int TME, int KW>
__device__ __forceinline__ void finish_tile(float16_t (&acc)[TME][TN], half_t* __restrict__ Y, const Epilogue& epilogue,
                                            int M, int N, int m0, int n0, unsigned char* lds_all, int set, int wave,
                                            int lane) {
  using Cfg = LdsGemmCfg<Policy, TM, TN, WM, WN, WPE>;
  const int wm = wave / WN, wn = wave % WN;
  unsigned char* stage = lds_all;
  if constexpr (KW == 2) {
    // set 1's sums in register order, 16 bytes per lane; behind them set 0's staging
    static_assert(!HalfStep<Policy>::value);
    constexpr int kSumBytes = 4 * TME * TN * 4096;
    static_assert(kSumBytes + 4 * RowwiseEpilogueCfg<TME, TN>::kBytesPerWave <= 2 * Cfg::kLdsBytes);
    float4_t* const sums = reinterpret_cast<float4_t*>(lds_all) + wave * (TME * TN * 256) + lane;
    __syncthreads();
    if (set == 1) {
#pragma unroll
      for (int i = 0; i < TME; ++i)
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            sums[((i * TN + t) * 4 + q) * 64] = float4_t{acc[i][t][4 * q], acc[i][t][4 * q + 1], acc[i][t][4 * q + 2], acc[i][t][4 * q + 3]};
    }
    __syncthreads();
    if (set == 1) return;
#pragma unroll
    for (int i = 0; i < TME; ++i)
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float4_t o = sums[((i * TN + t) * 4 + q) * 64];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][t][4 * q + e] += o[e];
        }
    stage = lds_all + kSumBytes;
  }

  // ---- epilogue ----
  // Row-wise through LDS (gemm_epilogue.h); each wavefront stages in a piece of its own.
  using ECfg = RowwiseEpilogueCfg<TME, TN>;
  static_assert(4 * ECfg::kBytesPerWave <= Cfg::kLdsBytes, "epilogue staging exceeds the ring");
  store_tile_rowwise<Epilogue, TME, TN>(acc, epilogue, Y, M, N, m0 + wm * TME * 32, n0 + wn * TN * 32,
                                        stage + wave * ECfg::kBytesPerWave, lane);
}

// One output tile of TME*32*WM rows x BN columns starting at (m0, n0).  TME is the
// number of 32-row sub-tiles per wavefront that are actually computed: TM for a full
// tile, TM/2 or TM/4 for the split tiles of the last, partially filled round.
//
// Schedule of one K-step (four phases kk = 0..3 of TME*TN MFMAs each).  Nothing but
// MFMAs may sit on the critical path of a wavefront that has its SIMD to itself, so
// every other instruction is slotted between them:
//   phases 0-2  per MFMA slot one LDS read of an activation fragment of phase kk+1 (the first
//               TME slots) and one half of the unpacking of a weight pair of phase kk+1 (bit
//               pattern in an early slot, arithmetic in a later one); in phase 0 also all direct
//               loads of step ks+2, one every few slots (the texture path accepts 64 B per cycle
//               and CU: issued in a burst they block the wavefront for hundreds of cycles);
//   phase 3     first s_waitcnt vmcnt (this wavefront's loads of step ks+1 have landed)
//               and s_barrier (everyone's have); then, between its MFMAs, the packed
//               weights, the first activation fragments and the first weight pairs of
//               step ks+1, so that step ks+1 starts multiplying at once.
// The K loop is one basic block: the loads past the last step are issued too, against a descriptor that holds nothing, so
// that the waits are constants (and leave the last of those loads on their way: the ring is drained behind the loop, in
// front of finish_tile).  Branches around them cost more than themselves, since the compiler moves the unpacking
// across the end of a block, behind the barrier.  With buffer loads, the integers of a pair finished in its first slot and
// no wait for the scale in front of phase 3: 540 -> 308 instructions per step, N = 22016, K = 4096, M = 8192 1292 -> 1207 us,
// int4 N = 28672, K = 8192, M = 500 232 -> 219 us, N = 11008, K = 4096, M = 200 36.4 -> 35.4 us.
//
// One barrier per K-step suffices (three slots shown): slot (ks+2)%3 = (ks-1)%3 is refilled by loads issued after
// the barrier of step ks-1, and every wavefront has waited for its last LDS reads of that slot
// (the phase-3 fragments of step ks-1) before that barrier.
//
// KW = 2: the workgroup has two sets of four wavefronts, each with a ring of its own; set 0 takes the first half of
// the K-steps, set 1 the second half (K % 128 == 0: as many steps, so as many barriers, in both), and set 1 hands
// its sums to set 0 through LDS.  For launches with no more tiles than CUs: a wavefront alone on its SIMD leaves the
// matrix core idle whenever it waits, and a second workgroup for the CU does not exist.
template <class Policy, class Epilogue, int TM, int TN, int WM, int WN, int WPE, int TME, int KW = 1>
__device__ __forceinline__ void gemm_lds_tile(const typename Policy::Args& wargs,
                                              const half_t* __restrict__ X, half_t* __restrict__ Y,
                                              const Epilogue& epilogue, int M, int N, int K, int m0,
                                              int n0, unsigned char* lds) {
  using Cfg = LdsGemmCfg<Policy, TM, TN, WM, WN, WPE>;
  constexpr int kALoadsE = Cfg::kALoads * TME / TM;  // direct A loads per wavefront per step
  constexpr int L = kALoadsE + Cfg::kBLoads + Cfg::kSLoads;  // direct loads per wavefront per step
  constexpr int NSLOT = TME * TN;                    // MFMAs per phase
  constexpr int NPAIR = TN * 4;                      // weight pairs to unpack per phase
  static_assert(kALoadsE >= 1, "tile too small to split further");
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  static_assert(KW == 1 || KW == 2);
  const int set = KW == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) - 4 * set;
  const int wm = wave / WN, wn = wave % WN;
  const int lj = lane & 31, lh = lane >> 5;
  const int ksteps = (K >> 6) / KW, ks0 = set * ksteps;  // this set's steps: ks0 .. ks0 + ksteps - 1
  unsigned char* const lds_all = lds;
  lds += set * Cfg::kLdsBytes;

  // ---- global sources of this lane's direct loads: buffer descriptors at the tile's first row and column, byte offsets
  //      from there (rows past M / N are clamped: they only feed accumulators that are never stored) ----
  const char* const a_base = reinterpret_cast<const char*>(X + (int64_t)m0 * K);
  using Off = std::conditional_t<Wide<Policy>::value, int64_t, uint32_t>;
  Off a_off[kALoadsE];
#pragma unroll
  for (int i = 0; i < kALoadsE; ++i) {
    const int s = (wave * kALoadsE + i) * 64 + lane;  // LDS chunk slot
    const int r = s >> 3, c = (s & 7) ^ WQ_SWZ(r);
    a_off[i] = (Off)(min(m0 + r, M - 1) - m0) * (Off)(2 * (int64_t)K) + c * 16;
  }
  const char* const b_base = Policy::b_src(wargs, n0, 0, N, K);
  Off b_off[Cfg::kBLoads];
#pragma unroll
  for (int i = 0; i < Cfg::kBLoads; ++i)
    b_off[i] = (Off)(Policy::b_src(wargs, n0, (wave * Cfg::kBLoads + i) * 64 + lane, N, K) - b_base);
  // scales staged per step (format A): 64 columns per wavefront (with BN = 128 wavefronts 2
  // and 3 repeat the loads of wavefronts 0 and 1)
  const char* s_base = b_base;
  Off s_off[2] = {0, 0};
  const int s_col = min(n0 + (wave * 64) % Cfg::BN + lane, N - 1);
  if constexpr (Cfg::kSLoads > 0) {
    s_base = Policy::s_src(wargs, n0, K);
    s_off[0] = (Off)(Policy::s_src(wargs, s_col, K) - s_base);
    if constexpr (Cfg::kSLoads == 2) s_off[1] = (Off)(Policy::s_src2(wargs, s_col, K) - s_base);
  }

  // direct load number idx (0 .. L-1) of this set's step ks into the slot at byte `slot` of the ring; past the last
  // step nothing is read, so that the loop has neither a branch nor a second form of its waits
  auto issue_one = [&](int ks, int slot, int idx) {
    unsigned char* const to = lds + slot;
    const int k = ks0 + ks;
    const bool is_a = idx < kALoadsE, is_b = !is_a && idx < kALoadsE + Cfg::kBLoads;
    const int i = is_a ? idx : is_b ? idx - kALoadsE : idx - kALoadsE - Cfg::kBLoads;
    unsigned char* const dst = to + (is_a   ? Cfg::kAOff + (wave * kALoadsE + i) * 1024
                                     : is_b ? Cfg::kBOff + (wave * Cfg::kBLoads + i) * 1024
                                            : Cfg::kSOff + i * (Cfg::BN * 4) + (wave * 64 % Cfg::BN) * 4);
    if constexpr (Wide<Policy>::value) {
      const int kc = min(k, ks0 + ksteps - 1);
      const char* const src = is_a   ? a_base + a_off[i] + (int64_t)kc * 128
                              : is_b ? b_base + b_off[i] + (int64_t)kc * Policy::kStepStride
                                     : s_base + s_off[i] + Policy::s_offset(wargs, kc);
      if (is_a || is_b) __builtin_amdgcn_global_load_lds((wq_gptr_t)src, (wq_lptr_t)dst, 16, 0, 0);
      else __builtin_amdgcn_global_load_lds((wq_gptr_t)src, (wq_lptr_t)dst, 4, 0, 0);
    } else {
      const int live = wq_live(ks, ksteps);
      if (is_a) direct_load16_if(live, a_base, (wq_lptr_t)dst, a_off[i], k * 128);
      else if (is_b) direct_load16_if(live, b_base, (wq_lptr_t)dst, b_off[i], k * Policy::kStepStride);
      else direct_load4_if(live, s_base, (wq_lptr_t)dst, s_off[i], (int)Policy::s_offset(wargs, k));
    }
  };

  float16_t acc[TME][TN];
#pragma unroll
  for (int i = 0; i < TME; ++i)
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][t][r] = 0.0f;

  typename Policy::Frag bw[TN];   // this lane's packed weights (and scale) of the step being unpacked
  typename Policy::Scale bs[TN];
  if (!Cfg::kSLoads) {
#pragma unroll
    for (int t = 0; t < TN; ++t) bs[t] = Policy::const_scale(wargs, min(n0 + (wn * TN + t) * 32 + lj, N - 1));
  }
  half8_t aop[2][TME], bop[2][TN];
  auto read_b = [&](const unsigned char* slot) {
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      const int n = (wn * TN + t) * 32 + lj;
      Policy::read(bw[t], slot + Cfg::kBOff, n, lh);
      if constexpr (Cfg::kSLoads == 2) bs[t] = Policy::read_scale2(slot + Cfg::kSOff + n * 4, Cfg::BN * 4, n, lh);
      else if (Cfg::kSLoads) bs[t] = Policy::read_scale(slot + Cfg::kSOff + n * 4, lh);
    }
  };
  int a_lane[4];  // fragment kk of row lj of a sub-tile, from the slot on (WQ_SWZ is the same for all sub-tiles)
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
    a_lane[kk] = Cfg::kAOff + (wm * TME * 32 + lj) * 128 + (((4 * lh + kk) ^ WQ_SWZ(lj)) << 4);
  auto read_a = [&](const unsigned char* slot, int kk, int i) {
    return *reinterpret_cast<const half8_t*>(slot + a_lane[kk] + i * 4096);
  };

  // ---- prologue: steps 0 .. kStages - 2 in flight, operands of step 0 ready ----
  constexpr int AHEAD = Cfg::kStages - 1;  // steps of loads in flight while a step is multiplied
  static_assert(AHEAD * L <= 63, "vmcnt holds 6 bits");
#pragma unroll
  for (int st = 0; st < AHEAD; ++st) {
#pragma unroll
    for (int idx = 0; idx < L; ++idx) issue_one(st, st * Cfg::kStageBytes, idx);
  }
  WQ_WAITCNT_VM((AHEAD - 1) * L);  // loads retire in order: step 0 has landed
  __builtin_amdgcn_s_barrier();
  read_b(lds);
#pragma unroll
  for (int i = 0; i < TME; ++i) aop[0][i] = read_a(lds, 0, i);
#pragma unroll
  for (int t = 0; t < TN; ++t) {
    half2_t d[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) d[j] = Policy::pair(bw[t], 0, j, bs[t]);
    bop[0][t] = half8_t{d[0].x, d[0].y, d[1].x, d[1].y, d[2].x, d[2].y, d[3].x, d[3].y};
  }

  // Phase 3 prepares the next step unconditionally: in the last step it reads a slot that
  // holds stale data and unpacks it for nobody.
  int at = 0, last = AHEAD * Cfg::kStageBytes;  // slots of step ks and of ks - 1, which takes step ks + AHEAD
  for (int ks = 0; ks < ksteps; ++ks) {
    const int next = at == AHEAD * Cfg::kStageBytes ? 0 : at + Cfg::kStageBytes;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int cur = kk & 1, nxt = cur ^ 1;
      const unsigned char* const a_from = lds + (kk == 3 ? next : at);  // activation fragments of the next phase
      const int a_kk = kk == 3 ? 0 : kk + 1;
      if (kk == 3) {
        // loads of step ks+1 landed (those of the later ones may be in flight), own LDS reads done
        WQ_WAITCNT_VM_LGKM0((AHEAD - 1) * L);
        __builtin_amdgcn_s_barrier();
        read_b(lds + next);
      }
      half2_t dq[TN][4];
      uint32_t pb[NPAIR];
      // Slots of the unpacking: the exact integers in the first half of the usable slots, the products in the
      // second half; in phase 3 the packed weights were requested from LDS just above, so the first slots stay free.
      const int first = kk < 3 ? 0 : NSLOT * 3 / 8, usable = NSLOT - first, half = usable / 2;
      if constexpr (ScalePerK<Policy>::value) {
#pragma unroll
        for (int t = 0; t < TN; ++t) Policy::phase_begin(bs[t], (kk + 1) & 3);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int sl = 0; sl < NSLOT; ++sl) {
        const int i = sl / TN, t = sl % TN;
        acc[i][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(aop[cur][i], bop[cur][t], acc[i][t], 0, 0, 0);
        // the activation fragments of the next phase, evenly
#pragma unroll
        for (int r = 0; r < TME; ++r)
          if (sl == r * TN + TN - 1) aop[nxt][r] = read_a(a_from, a_kk, r);
#pragma unroll
        for (int p = 0; p < NPAIR; ++p) {
          const int tt = p >> 2, j = p & 3;
          if (sl == first + p * half / NPAIR) pb[p] = Policy::pair_bits(bw[tt], (kk + 1) & 3, j);
          if (sl == first + half + p * (usable - half) / NPAIR) {
            if constexpr (ScalePerK<Policy>::value) dq[tt][j] = Policy::pair_finish_at(pb[p], bs[tt], j);
            else dq[tt][j] = Policy::pair_finish(pb[p], bs[tt]);
          }
        }
        // direct loads of step ks+AHEAD, all in phase 0 (into the slot of step ks-1, free since the
        // barrier of its phase 3): timed on the GPU, one phase with loads and three without beat
        // the same loads spread over two phases (by 1-2 %) or over all four (by 15 %)
        if (kk == 0) {
          const int l0 = sl * L / NSLOT, l1 = (sl + 1) * L / NSLOT;
#pragma unroll
          for (int idx = l0; idx < l1; ++idx) issue_one(ks + AHEAD, last, idx);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int t = 0; t < TN; ++t)
        bop[nxt][t] = half8_t{dq[t][0].x, dq[t][0].y, dq[t][1].x, dq[t][1].y,
                              dq[t][2].x, dq[t][2].y, dq[t][3].x, dq[t][3].y};
    }
    last = at;
    at = next;
  }

  // ---- the last 32 k of a K that is no multiple of 64: two MFMAs per sub-tile straight from global memory.
  // Once per tile, so it is not worth a place in the pipeline; the operands split k between the lane halves
  // like the MFMA does (both alike, so any split gives the same sum). ----
  if constexpr (HalfStep<Policy>::value) {
    const int k0 = ksteps << 6;
    half8_t b[TN][2];
#pragma unroll
    for (int t = 0; t < TN; ++t) Policy::half_step(wargs, min(n0 + (wn * TN + t) * 32 + lj, N - 1), k0, K, lh, b[t]);
#pragma unroll
    for (int i = 0; i < TME; ++i) {
      const half_t* const a = X + (int64_t)min(m0 + (wm * TME + i) * 32 + lj, M - 1) * K + k0 + 8 * lh;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const half8_t av = *reinterpret_cast<const half8_t*>(a + 16 * c);
#pragma unroll
        for (int t = 0; t < TN; ++t) acc[i][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, b[t][c], acc[i][t], 0, 0, 0);
      }
    }
  }

  if constexpr (ColumnScale<Policy>::value) {
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int i = 0; i < TME; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][t][r] *= (float)bs[t];
  }
  // The loads past the last step write to the ring like all others (zeros; in the wide form the last step again), and their
  // places overlap the pieces in which other wavefronts stage: all of them land before anyone goes on.
  WQ_WAITCNT_VM(0);
  __builtin_amdgcn_s_barrier();
  finish_tile<Policy, Epilogue, TM, TN, WM, WN, WPE, TME, KW>(acc, Y, epilogue, M, N, m0, n0, lds_all, set, wave, lane);
}

// The same tile with the weights in registers.  With the wavefronts of a workgroup side by side (WM = 1) nobody shares a
// wavefront's columns, so staging them in LDS buys nothing, and fetching them step by step is expensive: a format that
// is contiguous along K gives a step 32 bytes of codes and 4 of scales per column, and every load touches a cache line
// per column however little it takes of it (without the loads of the scales, 1 KB of the 41 KB of a step, N = 22016,
// K = 4096, M = 8192 took 1120 instead of 1233 us, without those of the activations 1101).  So the codes of two steps
// are requested together, one piece of a column behind the other, and the scales of four; the K loop is written out for four steps, which
// makes the registers of a step and its slot in LDS fixed, and the ring of four slots holds activations only, a step
// more ahead than with the weights in it.
//
// Order of the loads (all of a wavefront's loads retire in order, and the wait for the activations counts them): step ks
// requests the activations of step ks + 3 in phase 0, the scales of the next four steps in phase 1 where ks % 4 == 0, and in
// phase 3 of odd steps the weights of steps ks + 3 and ks + 4, whose registers it has just emptied.  The prologue issues
// its loads in the order that the steps before the first would have had.
//
// Such a policy provides besides pair_bits / pair_finish
//   kStepStride            bytes between the steps of a column, of which a lane takes 16
//   kFourScales            true: a scale per 32 k, contiguous along K, taken for four steps at a time;
//                          false: a pair of halves that serves two steps
//   b_base(args, n0, K)    where the columns from n0 on begin, b_lane(n, n0, lh, K) the lane's first piece from there
//   s_base(args, n0, K), s_lane(args, n, n0, K)   the same for the scales
//   s_step(args, ks)       bytes from there to the pair of step ks (not kFourScales)
// Measured with the K loop below it, start of that change / before / now: N = 22016, K = 4096, M = 8192 1307 / 1219 / 1191 us;
// N = 4096, K = 11008, M = 2048 194 / 187 / 178; N = 11008, K = 4096, M = 200 37.2 / 35.5 / 32.4; AutoGPTQ with a group of 128,
// 128 x 128 tiles, 36.2 / - / 26.6 us.  With two wavefronts above one another (WM = 2: shapes 13 and 14, which the choice by
// size does not take on 256 CUs) both fetch the same weights, and it is the faster form all the same (256 x 128, N = 4096,
// K = 11008, M = 1024 135 -> 120 us; 256 x 256, N = 11008, K = 4096, M = 1024 107 -> 98).  fpA_intB stays with LDS: its 128-byte units are whole lines there, eight a load
// (int8, N = 28672, K = 8192, M = 128: 84 us, in registers 88).
template <class Policy, class Epilogue, int TM, int TN, int WM, int WN, int WPE, int TME, int KW = 1>
__device__ __forceinline__ void gemm_rb_tile(const typename Policy::Args& wargs, const half_t* __restrict__ X,
                                             half_t* __restrict__ Y, const Epilogue& epilogue, int M, int N, int K, int m0,
                                             int n0, unsigned char* lds_all) {
  using Cfg = LdsGemmCfg<Policy, TM, TN, WM, WN, WPE>;
  constexpr int kA = Cfg::kALoads * TME / TM;  // direct loads per wavefront and step
  constexpr bool kFour = Policy::kFourScales;
  constexpr int kB2 = kFour ? 2 * TN : 3 * TN;        // loads to registers per two steps
  constexpr int NSLOT = TME * TN, NPAIR = TN * 4;
  static_assert(kA >= 1 && Cfg::kStages == 4);
  const int tid = threadIdx.x, lane = tid & 63;
  const int set = KW == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) - 4 * set;
  const int wm = wave / WN, wn = wave % WN;
  const int lj = lane & 31, lh = lane >> 5;
  const int ksteps = (K >> 6) / KW, ks0 = set * ksteps;
  unsigned char* const lds = lds_all + set * Cfg::kLdsBytes;

  const char* const a_base = reinterpret_cast<const char*>(X + (int64_t)m0 * K);
  uint32_t a_off[kA];
#pragma unroll
  for (int i = 0; i < kA; ++i) {
    const int s = (wave * kA + i) * 64 + lane;
    const int r = s >> 3, c = (s & 7) ^ WQ_SWZ(r);
    a_off[i] = (uint32_t)(min(m0 + r, M - 1) - m0) * (uint32_t)(2 * K) + c * 16;
  }
  const char* const b_base = Policy::b_base(wargs, n0, K);
  const char* const s_base = Policy::s_base(wargs, n0, K);
  uint32_t b_off[TN], s_off[TN];
#pragma unroll
  for (int t = 0; t < TN; ++t) {
    const int n = min(n0 + (wn * TN + t) * 32 + lj, N - 1);
    b_off[t] = Policy::b_lane(n, n0, lh, K);
    s_off[t] = Policy::s_lane(wargs, n, n0, K);
  }

  typename Policy::Frag bq[4][TN];  // the codes of four steps
  uint4_t s_cur[TN], s_next[TN];    // scales of this set of four steps and of the next (kFour)
  half2_t s_pair[2][TN];            // (not kFour)
  // past the last step: descriptors that hold nothing
  auto live = [&](int ks) { return wq_live(ks, ksteps); };
  auto issue_a = [&](int ks, int slot, int i) {
    direct_load16_if(live(ks), a_base, (wq_lptr_t)(lds + slot * Cfg::kStageBytes + (wave * kA + i) * 1024), a_off[i], (ks0 + ks) * 128);
  };
  auto load_b2 = [&](int ks, int slot, int idx) {  // what two steps need, idx 0 .. kB2 - 1
    if (idx < 2 * TN) {
      const int t = idx / 2, st = idx % 2;
      bq[slot + st][t].w = load_b128_if(live(ks + st), b_base, b_off[t], (ks0 + ks + st) * Policy::kStepStride);
    } else if constexpr (!kFour) {
      const int t = idx - 2 * TN;
      s_pair[slot >> 1][t] = as_half2(load_b32_if(live(ks), s_base, s_off[t], Policy::s_step(wargs, ks0 + ks)));
    }
  };
  // four steps' scales: the 8 from 2 ks on, or the last 8 of the row, moved down when they are taken over
  auto s_start = [&](int ks) { return min(2 * (ks0 + ks), (K >> 5) - 8); };
  auto load_s = [&](int ks, int t) {
    s_next[t] = load_b128_if(live(ks), s_base, s_off[t], 2 * s_start(ks));
  };
  auto take_s = [&](int ks, int t) {
    const int d = (2 * (ks0 + ks) - s_start(ks)) >> 1;
    uint4_t v = s_next[t];
    v = (d & 1) ? uint4_t{v.y, v.z, v.w, v.w} : v;
    s_cur[t] = (d & 2) ? uint4_t{v.z, v.w, v.w, v.w} : v;
  };
  auto scale_of = [&](int u, int t) {
    if constexpr (kFour) {
      const uint32_t w = u == 0 ? s_cur[t].x : u == 1 ? s_cur[t].y : u == 2 ? s_cur[t].z : s_cur[t].w;
      return as_half2(w >> (16 * lh)).x;
    } else {
      return s_pair[u >> 1][t];
    }
  };

  float16_t acc[TME][TN];
#pragma unroll
  for (int i = 0; i < TME; ++i)
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][t][r] = 0.0f;
  half8_t aop[2][TME], bop[2][TN];
  std::conditional_t<kFour, half_t, half2_t> sc[TN];
  // fragment kk of row lj of a sub-tile in slots 0 and 1, and in slots 2 and 3 (an LDS instruction reaches 64 KiB from its
  // address register; left to itself the compiler keeps a register for everything beyond, and spills)
  int a_lane[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      a_lane[h][kk] = set * Cfg::kLdsBytes + 2 * h * Cfg::kStageBytes + (wm * TME * 32 + lj) * 128 + (((4 * lh + kk) ^ WQ_SWZ(lj)) << 4);
      asm volatile("" : "+v"(a_lane[h][kk]));
    }
  auto read_a = [&](int slot, int kk, int i) {
    return *reinterpret_cast<const half8_t*>(lds_all + a_lane[slot >> 1][kk] + (slot & 1) * Cfg::kStageBytes + i * 4096);
  };

  // ---- prologue (the waits count on its order) ----
  auto first_a = [&](int st) {
#pragma unroll
    for (int i = 0; i < kA; ++i) issue_a(st, st, i);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto first_b2 = [&](int st) {
#pragma unroll
    for (int i = 0; i < kB2; ++i) load_b2(st, st, i);
    __builtin_amdgcn_sched_barrier(0);
  };
  if constexpr (kFour) {
#pragma unroll
    for (int t = 0; t < TN; ++t) load_s(0, t);
    __builtin_amdgcn_sched_barrier(0);
  }
  first_a(0);
  first_b2(0);
  first_a(1);
  first_a(2);
  first_b2(2);
  WQ_WAITCNT_VM(2 * kA + 2 * kB2);  // step 0's activations have landed
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < TME; ++i) aop[0][i] = read_a(0, 0, i);
#pragma unroll
  for (int t = 0; t < TN; ++t) {
    if constexpr (kFour) take_s(0, t);
    sc[t] = scale_of(0, t);
    half2_t d[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) d[j] = Policy::pair_finish(Policy::pair_bits(bq[0][t], 0, j), sc[t]);
    bop[0][t] = half8_t{d[0].x, d[0].y, d[1].x, d[1].y, d[2].x, d[2].y, d[3].x, d[3].y};
  }

  auto step = [&](int ks, auto u_) {
    constexpr int u = decltype(u_)::value, un = (u + 1) & 3;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int cur = kk & 1, nxt = cur ^ 1;
      if (kk == 3) {
        // The activations of step ks + 1 have landed.  Requested after them: those of two steps, the weights of two
        // steps, and the scales where a set of four was begun in this step or the two before.
        WQ_WAITCNT_VM_LGKM0(2 * kA + kB2 + (kFour && u != 3 ? TN : 0));
        __builtin_amdgcn_s_barrier();
      }
      half2_t dq[TN][4];
      uint32_t pb[NPAIR];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int sl = 0; sl < NSLOT; ++sl) {
        const int i = sl / TN, t = sl % TN;
        acc[i][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(aop[cur][i], bop[cur][t], acc[i][t], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < TME; ++r)  // the activation fragments of the next phase, evenly
          if (sl == r * TN + TN - 1) aop[nxt][r] = kk == 3 ? read_a(un, 0, r) : read_a(u, kk + 1, r);
        if (kk == 3 && sl == 0) {
#pragma unroll
          for (int tt = 0; tt < TN; ++tt) {
            if constexpr (kFour) {
              if (u == 3) take_s(ks + 1, tt);
            }
            sc[tt] = scale_of(un, tt);
          }
        }
        // the exact integers in the first half of the slots, the products in the second
#pragma unroll
        for (int p = 0; p < NPAIR; ++p) {
          const int tt = p >> 2, j = p & 3;
          if (sl == p * (NSLOT / 2) / NPAIR) pb[p] = Policy::pair_bits(bq[kk == 3 ? un : u][tt], (kk + 1) & 3, j);
          if (sl == NSLOT / 2 + p * (NSLOT - NSLOT / 2) / NPAIR) dq[tt][j] = Policy::pair_finish(pb[p], sc[tt]);
        }
        if (kk == 0) {
#pragma unroll
          for (int idx = sl * kA / NSLOT; idx < (sl + 1) * kA / NSLOT; ++idx) issue_a(ks + 3, (u + 3) & 3, idx);
        }
        if constexpr (kFour && u == 0) {
          static_assert(NSLOT >= TN);
          if (kk == 1 && sl < TN) load_s(ks + 4, sl);
        }
        if constexpr (u % 2 == 1) {
          if (kk == 3) {
#pragma unroll
            for (int idx = sl * kB2 / NSLOT; idx < (sl + 1) * kB2 / NSLOT; ++idx) load_b2(ks + 3, (u + 3) & 3, idx);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int t = 0; t < TN; ++t) {
        bop[nxt][t] = half8_t{dq[t][0].x, dq[t][0].y, dq[t][1].x, dq[t][1].y, dq[t][2].x, dq[t][2].y, dq[t][3].x, dq[t][3].y};
        // (or the compiler moves the unpacking into the next step, behind the test for the end)
        if (kk == 3) asm volatile("" : "+v"(bop[nxt][t]));
      }
    }
  };
  int ks = 0;
  for (; ks + 4 <= ksteps; ks += 4) {  // (one way out: with a test behind every step the sums change registers at the end)
    step(ks, std::integral_constant<int, 0>{});
    step(ks + 1, std::integral_constant<int, 1>{});
    step(ks + 2, std::integral_constant<int, 2>{});
    step(ks + 3, std::integral_constant<int, 3>{});
  }
  if (ks < ksteps) step(ks, std::integral_constant<int, 0>{});
  if (ks + 1 < ksteps) step(ks + 1, std::integral_constant<int, 1>{});
  if (ks + 2 < ksteps) step(ks + 2, std::integral_constant<int, 2>{});
  WQ_WAITCNT_VM(0);
  __builtin_amdgcn_s_barrier();  // nothing is on its way to the ring, and nobody reads it
  finish_tile<Policy, Epilogue, TM, TN, WM, WN, WPE, TME, KW>(acc, Y, epilogue, M, N, m0, n0, lds_all, set, wave, lane);
}

// Row slices (1, 2 or 4; 8 where the policy carries the extra copy of the tile body, `fine`) that the tiles of
// the last, partially filled round are cut into: as many as still run all at once.  (Every slice unpacks all
// columns of its tile, so slices get less efficient as they get lower: eight only pay on 32 tiles or fewer:
// M = 256, N = 4096, K = 11008 format A 73.6 -> 68.6 us.)  A rest that already has a CU per tile is only cut if every slice gets a
// CU of its own: two slices sharing a CU take as long as the whole tile, and read its weights twice.
inline int lds_tail_split(int rest, int slots, int cus, int TM, int a_loads, bool fine = false) {
  const int room = rest <= cus ? cus : slots;
  if (fine && TM % 8 == 0 && a_loads % 8 == 0 && rest * 8 <= room) return 8;
  for (int sp : {4, 2})
    if (TM % sp == 0 && a_loads % sp == 0 && rest * sp <= room) return sp;
  return 1;
}

// Relative duration of the LDS-staged GEMM on an M x N problem under tile configuration 11 (256 x 256
// tiles), 17 (128 x 128, two workgroups per CU) or 18 (256 x 128): rounds of the machine times tile
// area over the rate one CU sustains on such tiles.  The rates are tile areas per microsecond measured
// at K = 8192, N = 28672 with int8 weights (128 x 128 alone on its CU 193, two per CU 243 together;
// 256 x 128: 254; 256 x 256: 294); row slices of a cut tile run at 0.74 (halves) and 0.56 (quarters) of
// them (a slice unpacks all columns of its tile whatever its height; fitted to launches that are one cut round:
// N = 4096 .. 12288, M = 192 .. 1024, where 0.85 / 0.75 chose 256 x 256 tiles 10 .. 15 % too slow).  The model reproduces the measured times at M = 65 .. 2048 within 6 %.
//
// An epilogue with an activation (exp, erf) adds time that does not depend on K: per round 4 us (17), 18 us (18),
// 26 us (11) for whole tiles, less for slices.  Two workgroups per CU multiply through each other's epilogue, one
// cannot.  Fitted to silu and gelu over seven (N, K), K = 1024 .. 12288, M = 128 .. 2048: the choice is 0.2 % slower
// than the fastest on average and 6 % at most; without the term 10 % and 34 % (int8, N = 16384, K = 1024, M = 768:
// 64.8 -> 52.9 us; N = 28672, K = 2048, M = 1536: 288 -> 242 us; N = 22016, K = 4096, M = 512: 137 -> 124 us).
inline double lds_cfg_cost(int cfg, int64_t M, int64_t N, int64_t K, bool activates, int cus) {
  const int BM = cfg == 17 ? 128 : 256, BN = cfg == 11 ? 256 : 128, per_cu = cfg == 17 ? 2 : 1;
  const double rate_alone = cfg == 17 ? 193.0 : cfg == 18 ? 254.0 : 294.0;
  const double rate_full = cfg == 17 ? 243.0 : rate_alone;  // per CU, every slot taken
  const int64_t tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  const int slots = cus * per_cu;
  const int rest = (int)(tiles % slots);
  const double area = (double)BM * BN;
  const double fixed = activates ? (cfg == 17 ? 4.0 : cfg == 18 ? 18.0 : 26.0) * 8192.0 / (double)K : 0.0;
  double t = (double)(tiles / slots) * (per_cu * area / rate_full + fixed);
  if (rest) {
    const int split = lds_tail_split(rest, slots, cus, BM / 32, BM / 32);
    const bool alone = rest * split <= cus;
    const double slice = split == 4 ? 0.56 : split == 2 ? 0.74 : 1.0;
    t += area / split * (alone ? 1 : per_cu) / ((alone ? rate_alone : rate_full) * slice);
    t += fixed / split * (alone && cfg == 17 ? 0.7 : 1.0);
  }
  return t;
}

// Configuration 19: 128 x 128 tiles with the K-steps of a tile split between two sets of wavefronts (KW = 2), for
// launches that have no more such tiles than CUs.  Against the fastest of 17, 18 and 11: int8, K = 8192, N = 28672,
// M = 128 93 -> 85 us; K = 4096, N = 11008, M = 200 41.5 -> 35.2 us, int4 38.7 -> 32.8 us; N = K = 1024, M = 128
// 9.4 -> 7.9 us; over five such shapes, M = 70 .. 1024, 1 .. 28 %.  Slower at one of them only, int8, N = K = 8192,
// M = 100 .. 128 (55.0 -> 55.8 us: rows of weights a power of two apart, read by a row slice on every CU); its neighbours
// gain as elsewhere (N = 7936 53.2 -> 47.1, N = 8320 57.3 -> 42.8, K = 8320 53.8 -> 43.2 us), which leaves no rule to draw.
inline bool lds_k_halves(int64_t M, int64_t N, int64_t K, int cus) {
  return K % 128 == 0 && ((M + 127) / 128) * ((N + 127) / 128) <= cus;
}

// The same for 4-bit codes with a scale per group in front of the rule of choose_q4_lds_cfg, whose 256 x 128 tiles in
// row slices are as fast where they fill the machine: four or eight slices on 7/8 of the CUs (N = 4096, K = 11008:
// M = 256 69 against 73 us, M = 500 80 against 85), or tiles for 3/4 of them (N = 12288, K = 4096, M = 256 39.0
// against 39.5; N = 5120, K = 13824, M = 640 122 against 124).  A last row of tiles with hardly a row in it costs
// this form a whole tile too (N = 11008, K = 4096, M = 129: 38 against 39 us).  Elsewhere: N = 11008, K = 4096,
// M = 128 33.5 -> 29.7, M = 200 38.6 -> 36.3 us; N = 5120, K = 13824, M = 300 113 -> 93 us.
inline bool q4_lds_k_halves(int64_t M, int64_t N, int64_t K, int cus) {
  const int64_t tiles_n = (N + 127) / 128, tiles = ((M + 127) / 128) * tiles_n;
  if (K % 128 != 0 || tiles * 4 >= (int64_t)cus * 3 || (M - 1) % 128 < 15) return false;
  const int64_t rest = ((M + 255) / 256) * tiles_n;  // fewer than 3/4 of the CUs, as well
  const int split = lds_tail_split((int)rest, cus, cus, 8, 8, true);
  const int64_t slices = tiles_n * ((M * split + 255) / 256);
  return !(M > 128 && split >= 4 && slices * 8 >= (int64_t)cus * 7);
}

// Policy::kFineTail = true: the kernels of that policy also hold the tile body for slices of TM / 8 sub-tiles.
template <class P, class = void>
struct FineTail : std::false_type {};
template <class P>
struct FineTail<P, std::void_t<decltype(P::kFineTail)>> : std::bool_constant<P::kFineTail> {};

template <class Policy, class Epilogue, int TM, int TN, int WM, int WN, int WPE, int TME, int KW>
__device__ __forceinline__ void gemm_tile(const typename Policy::Args& wargs, const half_t* __restrict__ X,
                                          half_t* __restrict__ Y, const Epilogue& epilogue, int M, int N, int K, int m0,
                                          int n0, unsigned char* lds) {
  if constexpr (RegB<Policy>::value)
    gemm_rb_tile<Policy, Epilogue, TM, TN, WM, WN, WPE, TME, KW>(wargs, X, Y, epilogue, M, N, K, m0, n0, lds);
  else
    gemm_lds_tile<Policy, Epilogue, TM, TN, WM, WN, WPE, TME, KW>(wargs, X, Y, epilogue, M, N, K, m0, n0, lds);
}

// Workgroup -> work item.  The first n_full workgroups compute whole tiles (as many
// as fill complete rounds of the machine); the tiles of the last, partially filled
// round are cut into `split` row slices of TM/split sub-tiles so that the round is
// shorter instead of leaving most CUs idle while a few finish whole tiles.
template <class Policy, class Epilogue, int TM, int TN, int WM, int WN, int WAVES_PER_EU, int KW>
__global__ __launch_bounds__(256 * KW) __attribute__((amdgpu_waves_per_eu(WAVES_PER_EU, WAVES_PER_EU)))
void gemm_lds_kernel(typename Policy::Args wargs, const half_t* __restrict__ X, half_t* __restrict__ Y,
                     Epilogue epilogue, int M, int N, int K, int tiles_m, int tiles_n, int n_full,
                     int split, int group_m) {
  using Cfg = LdsGemmCfg<Policy, TM, TN, WM, WN, WAVES_PER_EU>;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  // Tiles are numbered in bands of group_m rows of tiles, N-fastest inside a band and M-fastest inside a column of
  // the band, and workgroups go to the XCDs round-robin: XCD x (own L2) takes a contiguous range of that order,
  // so the tiles it runs at one time are group_m tiles high and share their activation rows and weight columns
  // through its L2.  The same for the slices of the last, partial round.
  auto tile_of = [&](int t, int& tile_m, int& tile_n) {
    const int width = group_m * tiles_n, band = t / width, in_band = t - band * width;
    const int first_m = band * group_m, rows = min(group_m, tiles_m - first_m);
    tile_m = first_m + in_band % rows;
    tile_n = in_band / rows;
  };
  int pid = blockIdx.x;
  if (pid < n_full) {
    const int per = n_full / 8, rem = n_full % 8;
    const int xcd = pid & 7, idx = pid >> 3;
    int tile_m, tile_n;
    tile_of(xcd * per + min(xcd, rem) + idx, tile_m, tile_n);
    gemm_tile<Policy, Epilogue, TM, TN, WM, WN, WAVES_PER_EU, TM, KW>(wargs, X, Y, epilogue, M, N, K,
                                                        tile_m * Cfg::BM, tile_n * Cfg::BN, lds);
    return;
  }
  int q = pid - n_full;
  if (n_full > 0) {  // (a launch of one partial round keeps the plain order: measured 2-3 % faster there)
    const int slices = ((int)gridDim.x - n_full), per = slices / 8, rem = slices % 8;
    const int xcd = q & 7, idx = q >> 3;  // n_full is a multiple of the CU count: the XCD of this workgroup is q mod 8
    q = xcd * per + min(xcd, rem) + idx;
  }
  const int part = q % split;
  int tile_m, tile_n;
  tile_of(n_full + q / split, tile_m, tile_n);
  const int m0 = tile_m * Cfg::BM + part * (Cfg::BM / split), n0 = tile_n * Cfg::BN;
  if (m0 >= M) return;  // a slice that lies entirely past the last row
  if (split == 2) {
    if constexpr (TM % 2 == 0)
      gemm_tile<Policy, Epilogue, TM, TN, WM, WN, WAVES_PER_EU, TM / 2, KW>(wargs, X, Y, epilogue, M, N, K, m0, n0, lds);
  } else if (split == 4) {
    if constexpr (TM % 4 == 0)
      gemm_tile<Policy, Epilogue, TM, TN, WM, WN, WAVES_PER_EU, TM / 4, KW>(wargs, X, Y, epilogue, M, N, K, m0, n0, lds);
  } else if (split == 8) {
    if constexpr (TM % 8 == 0 && FineTail<Policy>::value)
      gemm_tile<Policy, Epilogue, TM, TN, WM, WN, WAVES_PER_EU, TM / 8, KW>(wargs, X, Y, epilogue, M, N, K, m0, n0, lds);
  } else {
    gemm_tile<Policy, Epilogue, TM, TN, WM, WN, WAVES_PER_EU, TM, KW>(wargs, X, Y, epilogue, M, N, K, m0, n0, lds);
  }
}

template <class Policy, class Epilogue, int TM, int TN, int WM, int WN, int WPE, int KW = 1>
static int launch_gemm_lds(const char* who, const typename Policy::Args& wargs, const uint16_t* x,
                           uint16_t* y, const Epilogue& ep, int64_t M, int64_t N, int64_t K,
                           hipStream_t stream) {
  using Cfg = LdsGemmCfg<Policy, TM, TN, WM, WN, WPE>;
  WQ_REQUIRE(Wide<Policy>::value || K < kLdsGemmMaxK, "%s: internal: K=%lld needs 64-bit addresses", who, (long long)K);
  const int tiles_m = (int)((M + Cfg::BM - 1) / Cfg::BM);
  const int tiles_n = (int)((N + Cfg::BN - 1) / Cfg::BN);
  auto kern = gemm_lds_kernel<Policy, Epilogue, TM, TN, WM, WN, WPE, KW>;
  static DynamicLdsLimit limit;
  WQ_HIP(limit.ensure(reinterpret_cast<const void*>(kern), KW * Cfg::kLdsBytes));
  // Whole rounds of the machine run whole tiles; the tiles of the last, partial
  // round are cut into 2 or 4 row slices when that lets them all run at once.
  const int per_cu = std::max(1, std::min(WPE / KW, (160 * 1024) / (KW * Cfg::kLdsBytes)));
  const int slots = cu_count() * per_cu;
  const int total = tiles_m * tiles_n;
  const int n_full = (total / slots) * slots;
  const int rest = total - n_full;
  const int split = tuning().gemm_tail_split ? lds_tail_split(rest, slots, cu_count(), TM, Cfg::kALoads, FineTail<Policy>::value) : 1;
  // height of the block of tiles an XCD runs at one time: the activation rows of a tile against its weight
  // columns, in bytes per step of K, decide how a block of slots / 8 tiles is best shaped
  const double ratio = (double)(Cfg::BN * Policy::kColBytes) / (double)(Cfg::BM * 128);
  const double want = std::sqrt((double)(slots / 8) * ratio);
  int group_m = 1;
  while (group_m * 1.5 < want) group_m *= 2;
  group_m = std::max(1, std::min(group_m, tiles_m));
  if (n_full == 0) group_m = tiles_m;  // one partial round: M-fastest, workgroup i takes slice i
  WQ_LAUNCH(who, kern, dim3((unsigned)(n_full + rest * split)), dim3(256 * KW), KW * Cfg::kLdsBytes, stream, wargs,
            (const half_t*)x, (half_t*)y, ep, (int)M, (int)N, (int)K, tiles_m, tiles_n, n_full, split, group_m);
  return WQ_OK;
}

}  // namespace wq
#endif  // RELAX_AMD_CSRC_MFMA_GEMM_LDS_H_
