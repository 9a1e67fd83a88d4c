// MFMA GEMM whose matrix waves are fed by others (fed_gemm): tiles of up to 256 x 128, 160 x 192 or 128 x 256, of
// any output and contraction, for launches that give a CU one workgroup.
#pragma once
#include "gemm_solo.h"

namespace axn {
namespace {

// Stages that fit into a CU's LDS, at most five.
template <int BM, int BN>
constexpr int kFedStages = 163840 / ((BM + BN) * 128) < 5 ? 163840 / ((BM + BN) * 128) : 5;
template <int BM, int BN>
constexpr size_t kFedLds = (size_t)kFedStages<BM, BN> * (BM + BN) * 128;

// Eight waves, two on a SIMD: waves 0 .. 3 are solo_gemm's, a quarter of the tile each (BM / 2 x BN / 2), but copy
// nothing; waves 4 .. 7 do nothing but bring the operand tiles into LDS.  What bounds solo_gemm on tiles this small
// is that its one wave on a SIMD issues everything in order: a copy waits for its place in the CU's way to LDS (64
// bytes a clock; 256 x 128 tiles ask for 48 of them), and the MFMAs behind it wait with it.  Here only the copying
// waves wait.  The wave tile of half the registers is what leaves room for a second wave on a SIMD.
//   us of one round of 256 workgroups, contraction 4096, operands in the caches / from HBM:
//     256 x 128 tiles   solo_gemm 60.0 / 64.7   here 52.5 / 59.7
//     128 x 128 tiles             36.1 / 48.0        30.4 / 39.1
//   That is a forward's whole round alone.  Between other launches, and over the sizes that take 256 x 128 tiles, solo_gemm is
//   2 to 4 % ahead of this on them (gemm_*_rest_kernel); FED_256x128 runs where its own estimate is ahead (kFedTiles).
//   Without its copies this kernel takes 43 us on 256 x 128 tiles, its copies alone 37 / 55: from HBM they are the bound.
//   One, two or four copying waves, reads from the first or the fifth MFMA of a step on, s_setprio: all the same.
//
// LDS is a ring of whole stages (A tile, B tile), as many as fit.  The copying waves run ahead by all but one of them:
//   copying: stages 0 .. n-1; wait for stage 0; barrier;
//            for every stage p: wait for stage p + 1; barrier p; copy stage p + n into the slot of stage p
//   matrix : barrier; reads of (0, 0);
//            for every stage p: wait for its reads; MFMAs of step 0 | reads of (p, 1); wait; barrier p;
//                               MFMAs of step 1 | reads of (p + 1, 0)
// At barrier p every matrix wave holds the last fragments of stage p in registers, so its slot is free, and stage
// p + 1 has landed.  The sums' order is solo_gemm's: the two give the same bits.
//
// The operands' bounds are those of solo_gemm's EDGE (any contraction and operand size) throughout: they cost nothing
// here, the copying waves have time for them.  EDGE: the output's (false: whole tiles, rows 16-byte aligned).
// ODD, EPI_PAIR: as there.  ROUNDS: the workgroup takes tiles blockIdx.x, + gridDim.x, ... one after the other; the
// stages of all of them are one sequence to the waves and the ring (gridDim.x is a multiple of the XCDs' number); the output's
// columns are a multiple of 8 (the others go through LDS, which the next tile's stages have).
template <int BM, int BN, bool A_KMAJOR, bool B_KMAJOR, int EPI, bool OUT_F32, bool HALF, bool EDGE = true, bool ODD = false,
          bool ROUNDS = false>
__device__ __forceinline__ void fed_gemm(const GemmArgs& g) {
  constexpr uint32_t kOutside = 0x80000000u;
  constexpr int FRM = BM / 32, FRN = BN / 32, PK = 64, NM = FRM * FRN, NFRAG = FRM + FRN;
  constexpr int NST = kFedStages<BM, BN>;
  using OA = DeepOperand<A_KMAJOR, false, BM>;
  using OB = DeepOperand<B_KMAJOR, true, BN>;
  constexpr uint32_t STAGE = OA::BYTES + OB::BYTES;
  constexpr int NCA = OA::DMA_N, NCB = OB::DMA_N, NC = NCA + NCB;   // copies per stage and copying wave
  constexpr bool PAIR = EPI == EPI_PAIR, SWIGLU = EPI == EPI_SWIGLU;
  constexpr int READ_EVERY = NM / NFRAG >= 2 ? 2 : 1;   // a fragment read every .. MFMAs, from a step's first on
  static_assert(BM % 32 == 0 && BN % 64 == 0 && NM >= NFRAG, "blocks of a wave, and a place for every read in a step");
  static_assert(4 * NM + 8 * NFRAG <= 232, "accumulators and two sets of fragments leave room for addresses");
  static_assert(NST >= 3 && (NST - 1) * NC <= 63, "the count of a wait has six bits");
  static_assert(!PAIR || (A_KMAJOR && !B_KMAJOR), "the two-term product is the dgrad layout");
  static_assert(!ODD || (A_KMAJOR && B_KMAJOR), "the forward");
  static_assert(!ROUNDS || (!A_KMAJOR && !B_KMAJOR && EPI == AXN_EPI_NONE), "weight gradients: their epilogue needs no LDS");
  static_assert(!SWIGLU || (BN % 128 == 0 && A_KMAJOR && B_KMAJOR && !OUT_F32), "gate and up rows of a wave column");

  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & 63;
  const int wave8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = wave8 & 3;

  int tm, tn, split = 0;
  {
    int pid = blockIdx.x;
    if (g.splits > 1) {
      split = pid / (g.tiles_m * g.tiles_n);
      pid -= split * (g.tiles_m * g.tiles_n);
    }
    tile_of_workgroup(pid, g.tiles_m, g.tiles_n, tm, tn);
  }
  [[maybe_unused]] int tile = blockIdx.x;   // ROUNDS
  int m0 = tm * BM, n0 = tn * (SWIGLU ? BN / 2 : BN);
  const StageRange part = stages_of_part(g.Kc, split, g.splits);
  const int s0 = part.first, KP = part.count;
  const int rounds = ROUNDS ? (g.tiles_m * g.tiles_n - tile + (int)gridDim.x - 1) / (int)gridDim.x : 1;
  const int all = rounds * KP;   // stages
  [[maybe_unused]] auto next_tile = [&]() {
    tile += gridDim.x;
    tile_of_workgroup(tile, g.tiles_m, g.tiles_n, tm, tn);
    m0 = tm * BM;
    n0 = tn * BN;
  };

  if (wave8 >= 4) {
    OperandWalk wa, wb, wb2;   // (wb2: SWIGLU, the up weights')
    const int kfirst = PAIR ? g.k_first : g.Kc;
    wa.start(g.A, A_KMAJOR, g.M, kfirst, g.lda, m0, s0 * PK);
    wb.start(g.B, B_KMAJOR, g.N, kfirst, g.ldb, n0, s0 * PK);
    if constexpr (SWIGLU) wb2.start(g.B2, B_KMAJOR, g.N, g.Kc, g.ldb, n0, s0 * PK);
    // per-lane offsets of the copies: one and a stride (K-major), or one for each copy
    uint32_t ais = 0, bis = 0, va[A_KMAJOR ? 1 : NCA], vb[B_KMAJOR ? 1 : NCB];
    if constexpr (A_KMAJOR) {
      va[0] = OA::dma_offset(g.lda, 0, wave, lane, ais);
    } else {
#pragma unroll
      for (int i = 0; i < NCA; ++i) va[i] = OA::mnmajor_copy(g.lda, wave, lane, i);
    }
    if constexpr (B_KMAJOR) {
      vb[0] = OB::dma_offset(g.ldb, 0, wave, lane, bis);
    } else {
#pragma unroll
      for (int i = 0; i < NCB; ++i) vb[i] = OB::mnmajor_copy(g.ldb, wave, lane, i);
    }
    const int over = (int)((int64_t)(s0 + KP) * PK - g.Kc);   // contraction elements the last stage lacks
    uint32_t slot = 0;
    int next = 0;   // the stage to copy
    auto copy_stage = [&]() {
      if constexpr (ROUNDS)
        if (next == KP) {
          next_tile();
          wa.start(g.A, A_KMAJOR, g.M, kfirst, g.lda, m0, 0);
          wb.start(g.B, B_KMAJOR, g.N, kfirst, g.ldb, n0, 0);
          next = 0;
        }
      if (PAIR && (s0 + next) * PK == g.k_first) {
        wa.start(g.A2, A_KMAJOR, g.M, g.Kc - g.k_first, g.lda, m0, 0);
        wb.start(g.B2, B_KMAJOR, g.N, g.Kc - g.k_first, g.ldb, n0, 0);
      }
      if (over > 0 && next == KP - 1) {   // the last stage: chunks behind the contraction's end are zeros
        if (A_KMAJOR && 8 * OA::dma_chunk(wave, lane) >= PK - over) va[0] = kOutside;
        if (B_KMAJOR && 8 * OB::dma_chunk(wave, lane) >= PK - over) vb[0] = kOutside;
      }
      const __amdgpu_buffer_rsrc_t ra = wa.resource(), rb = wb.resource();
      [[maybe_unused]] __amdgpu_buffer_rsrc_t rb2 = rb;
      if constexpr (SWIGLU) {
        rb2 = wb2.resource();
        wb2.advance();
      }
      char* at = lds + slot;
      static_for<NCA>([&](auto c) {
        constexpr int I = decltype(c)::value;
        if constexpr (A_KMAJOR) OA::template dma_one<I>(ra, va[0], 0, ais, at, wave);
        else OA::template dma_one<I, 0>(ra, va[I], 0, 0, at, wave);
      });
      static_for<NCB>([&](auto c) {
        constexpr int I = decltype(c)::value;
        if constexpr (SWIGLU) {
          constexpr GateUpCopy from = gate_up_copy(BN, I);
          OB::template dma_one<I, from.at>(from.up ? rb2 : rb, vb[0], 0, bis, at + OA::BYTES, wave);
        } else if constexpr (B_KMAJOR) OB::template dma_one<I>(rb, vb[0], 0, bis, at + OA::BYTES, wave);
        else OB::template dma_one<I, 0>(rb, vb[I], 0, 0, at + OA::BYTES, wave);
      });
      wa.advance();
      wb.advance();
      slot = slot + STAGE == NST * STAGE ? 0 : slot + STAGE;
      ++next;
    };
    const int ahead = all < NST ? all : NST;
#pragma unroll 1
    for (int p = 0; p < ahead; ++p) copy_stage();
    if (all >= NST) wait_vmcnt<(NST - 1) * NC>();
    else wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
#pragma unroll 1
    for (int p = NST; p < all; ++p) {
      wait_vmcnt<(NST - 2) * NC>();   // all but the youngest NST - 2 stages have landed
      __builtin_amdgcn_s_barrier();
      copy_stage();
    }
    wait_vmcnt<0>();
#pragma unroll 1
    for (int p = 1; p < ahead; ++p) __builtin_amdgcn_s_barrier();
    return;
  }

  const int wm = wave >> 1, wn = wave & 1;
  f32x4 acc[FRM][FRN];
  const uint32_t lds0 = (uint32_t)(uintptr_t)LDS_PTR(char, lds);
  uint32_t ra0[OA::NADDR], rb0[OB::NADDR];
  OA::read_bases(ra0, wm * (BM / 2), lane);
  OB::read_bases(rb0, wn * (BN / 2), lane);
#pragma unroll
  for (int i = 0; i < OA::NADDR; ++i) ra0[i] += lds0;
#pragma unroll
  for (int i = 0; i < OB::NADDR; ++i) rb0[i] += lds0 + OA::BYTES;
#pragma unroll
  for (int i = 0; i < FRM; ++i)
#pragma unroll
    for (int j = 0; j < FRN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < FRM; ++i) tie_accumulators(acc[i]);

  bf16x8 fa0[FRM], fb0[FRN], fa1[FRM], fb1[FRN];  // register sets of steps 0 / 1
  // fragment f of FRM + FRN (A fragments, then B fragments) of step ST of the stage in the slot at s
  auto read = [&](auto st_, auto f_, uint32_t s) {
    constexpr int ST = decltype(st_)::value, f = decltype(f_)::value;
    bf16x8(&fa)[FRM] = ST ? fa1 : fa0;
    bf16x8(&fb)[FRN] = ST ? fb1 : fb0;
    if constexpr (f < FRM) {
      uint32_t ra[OA::NADDR];
#pragma unroll
      for (int i = 0; i < OA::NADDR; ++i) ra[i] = ra0[i] + s;
      OA::template read_frag<ST, f>(fa[f], ra);
    } else {
      uint32_t rb[OB::NADDR];
#pragma unroll
      for (int i = 0; i < OB::NADDR; ++i) rb[i] = rb0[i] + s;
      OB::template read_frag<ST, f - FRM>(fb[f - FRM], rb);
    }
  };
  uint32_t s = 0;
  auto stage = [&](auto last_) {
    constexpr bool LAST = decltype(last_)::value;
    const uint32_t sn = s + STAGE == NST * STAGE ? 0u : s + STAGE;
    static_for<2>([&](auto st_) {
      constexpr int ST = decltype(st_)::value;
      bf16x8(&fa)[FRM] = ST ? fa1 : fa0;
      bf16x8(&fb)[FRN] = ST ? fb1 : fb0;
      wait_all_fragments(fa, fb);   // every read of this set was issued during the previous step
      if constexpr (ST == 1 && !LAST) __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      static_for<NM>([&](auto m_) {
        constexpr int m = decltype(m_)::value;
        constexpr int i = m / FRN, j = m % FRN;
        // (register classes pinned and hazards as in solo_gemm; an accumulator is touched again NM - 1 MFMAs later)
        if constexpr (HALF)
          asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(fb[j]), "v"(fa[i]));
        else
          asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(fb[j]), "v"(fa[i]));
        if constexpr (m % READ_EVERY == 0 && m / READ_EVERY < NFRAG) {
          if constexpr (ST == 0) read(std::integral_constant<int, 1>{}, std::integral_constant<int, m / READ_EVERY>{}, s);
          else if constexpr (!LAST) read(std::integral_constant<int, 0>{}, std::integral_constant<int, m / READ_EVERY>{}, sn);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    });
    s = sn;
  };
  __builtin_amdgcn_s_barrier();
  static_for<NFRAG>([&](auto f_) { read(std::integral_constant<int, 0>{}, f_, s); });
  if constexpr (ROUNDS) {
#pragma unroll 1
    for (int r = 1; r < rounds; ++r) {
#pragma unroll 1
      for (int p = 0; p < KP; ++p) stage(std::false_type{});
      wait_all_fragments(fa0, fb0);   // the next tile's first: the stores' code may move registers
      asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
      for (int i = 0; i < FRM; ++i) tie_accumulators(acc[i]);
      store_blocks<EPI, OUT_F32, HALF, EDGE, ODD, false>(acc, g, 0, m0 + wm * (BM / 2), n0 + wn * (BN / 2), lane, nullptr);
#pragma unroll
      for (int i = 0; i < FRM; ++i) {
#pragma unroll
        for (int j = 0; j < FRN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        tie_accumulators(acc[i]);
      }
      next_tile();
    }
  }
#pragma unroll 1
  for (int p = 0; p < KP - 1; ++p) stage(std::false_type{});
  stage(std::true_type{});
  // (the accumulators pass through statements that follow the last MFMA by more than its latency, as in solo_gemm)
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int i = 0; i < FRM; ++i) tie_accumulators(acc[i]);
  if constexpr (SWIGLU) {
    store_gate_up<HALF, EDGE>(acc, g, m0 + wm * (BM / 2), n0 + wn * (BN / 4), lane);
  } else {
    // (s is the slot behind the last stage's: no wave reads or fills it any more)
    constexpr bool APART = EPI != AXN_EPI_NONE && !PAIR;
    store_blocks<EPI, OUT_F32, HALF, EDGE, ODD, APART>(acc, g, split, m0 + wm * (BM / 2), n0 + wn * (BN / 2), lane,
                                                       (float*)(lds + s) + wave * (FRM * 16 * 8));
  }
}

}  // namespace
}  // namespace axn
